// f32 batched matrix product (attention scores and contexts of a transformer encoder; op::v0::Dot on
// two matrices is the batch of one).  64 x 64 output tiles, the reduction in stages of 64 through
// LDS (f32), every wavefront a 32 x 32 quarter as 2 x 2 blocks of v_mfma_f64_16x16x4_f64.  The reference accumulates
// f32 products in double, k ascending (src/ngraph/runtime/reference/dot.hpp:34-37 with widen<float> =
// double, convolution.hpp:34-44), and rounds the sum to f32 once.  A product of two floats is exact
// in double, so a fused multiply-add rounds exactly as the reference's separate multiply and add;
// and the f64 matrix instruction accumulates its four products as a chain of such multiply-adds in
// k order (checked on the device against the chain: a million outputs over uniform, wide-range,
// integer-valued and cancelling operands, no bit differed -- and every parity test of this kernel
// is bit-exact against the oracle's sequential sum): the results are the reference's bit for bit.
// Operands are converted to double as fragments, one element a lane and matrix instruction, which
// is what makes the matrix instruction pay: the vector form converts eight operands for sixteen
// multiply-adds and is bound by the conversions.
#include <algorithm>

#include "hipq_common.h"
#include "hipq_quant_math.h"
#include "hipq_row_math.h"

namespace hipq
{
    namespace
    {
        typedef float f4 __attribute__((ext_vector_type(4)));
        typedef double d4 __attribute__((ext_vector_type(4)));
        constexpr int TM = 64, TN = 64, TK = 64, TKS = 16; // a stage is TK of the reduction, fetched and laid into LDS in pieces of TKS

        // where the matrices of batch element (outer, inner) start and how far apart their rows are (in
        // elements): the plain op has one batch level and dense matrices; views of a larger tensor
        // (the heads of a fused QKV projection, a context written head-interleaved) have two
        struct MatView
        {
            int64_t batch_inner;
            int64_t a_outer, a_inner, lda;
            int64_t b_outer, b_inner, ldb;
            int64_t o_outer, o_inner, ldo;
        };
        struct MatQuant
        {
            void* out; // null: none
            const float* scale;
            const void* zero_point;
            int32_t quant_t, mode;
        };

        // out[b] = op(A[b]) * op(B[b]): A is [M][K] (or [K][M] with ta), B is [K][N] (or [N][K] with tb).
        // A workgroup walks tiles item, item + grid, ...; the operands of the next stage -- the next
        // tile's first one after a tile's last -- are on their way into registers while this stage
        // multiplies, and a tile's stores drain under the next tile's products.  (One tile a workgroup,
        // all resident at once, runs the whole grid in lockstep: everyone loads, then everyone
        // multiplies, then everyone stores, and the three times add up.)
#ifndef BMM_PER_CU
#define BMM_PER_CU 3
#endif
#ifndef BMM_OCC
#define BMM_OCC __attribute__((amdgpu_waves_per_eu(3, 3)))
#endif
        struct TileAt
        {
            const float* A;
            const float* B;
            int64_t o_base;
            int m0, n0;
        };

        // WHOLE: every tile is full (M, N multiples of 64, K of TK) and every row 16-byte aligned, so
        // fetches and stores carry no bounds checks or scalar alternatives (uniform, chosen by the host)
        template <bool WHOLE, bool ta, bool tb>
        __global__ __launch_bounds__(256) BMM_OCC void batch_matmul_f32_kernel(const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ out, MatView view, MatQuant mq, int32_t M,
                                                                       int32_t K, int32_t N, int32_t m_tiles, int32_t n_tiles, int32_t tiles, int32_t vec_a, int32_t vec_b)
        {
            // An operand lies in LDS the way it lies in memory, so that every piece goes in as one 16-byte
            // write: [row][k] when its rows run along the reduction (A as given, B transposed), [k][row]
            // otherwise.  The pitches spread a fragment read (16 rows x 4 consecutive k a wavefront)
            // over all 64 banks: 68 floats a row ([row][k]: bank 4 row + k), 80 floats a k ([k][row]: bank 16 k + row).
            constexpr int PR = TK + 4, PK = TM + 16;
            constexpr int OPERAND = TM * PR > TK * PK ? TM * PR : TK * PK;
            __shared__ __attribute__((aligned(16))) float as[OPERAND];
            __shared__ __attribute__((aligned(16))) float bs[OPERAND];
            auto a_at = [](int k, int m) { return ta ? k * PK + m : m * PR + k; };
            auto b_at = [](int k, int n) { return tb ? n * PR + k : k * PK + n; };
            const int tid = threadIdx.x;
            const int64_t lda = view.lda, ldb = view.ldb, ldo = view.ldo;
            const int lane = tid & 63, wave = tid >> 6;
            const int r16 = lane & 15, kq = lane >> 4;          // fragment element: row / column r16 of a block, k = 4 * step + kq
            const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32; // this wavefront's quarter of the tile
            // workgroups are dealt round-robin to the 8 XCDs (an L2 each): renumbered so that
            // neighbouring tiles, which share operand rows, meet in one L2
            const int grid = static_cast<int>(gridDim.x);
            const int item = (grid & 7) == 0 ? (static_cast<int>(blockIdx.x) & 7) * (grid >> 3) + (static_cast<int>(blockIdx.x) >> 3) : static_cast<int>(blockIdx.x);
            const uint32_t batch_inner = static_cast<uint32_t>(view.batch_inner < (1ll << 31) ? view.batch_inner : (1ll << 31)); // (there are fewer than 2^31 tiles)
            auto tile_at = [&](int t) -> TileAt {
                const int nt = t % n_tiles;
                t /= n_tiles;
                const int mt = t % m_tiles;
                const uint32_t batch = static_cast<uint32_t>(t / m_tiles);
                const int64_t bo = batch / batch_inner, bi = batch - bo * batch_inner; // (32-bit division)
                return TileAt{a + bo * view.a_outer + bi * view.a_inner, b + bo * view.b_outer + bi * view.b_inner, bo * view.o_outer + bi * view.o_inner, mt * TM, nt * TN};
            };
            // 64 x 16 elements of each operand a piece, four a lane, contiguous along the operand's rows in memory
            auto fetch_a = [&](const TileAt& w, int k0) -> f4 {
                f4 v = f4{0.0f, 0.0f, 0.0f, 0.0f};
                if (!ta)
                {
                    const int r = tid >> 2, kq = (tid & 3) * 4; // A[m0 + r][k0 + kq ..]
                    if (WHOLE || (vec_a && w.m0 + r < M && k0 + kq + 3 < K))
                        v = *reinterpret_cast<const f4*>(w.A + static_cast<int64_t>(w.m0 + r) * lda + k0 + kq);
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[i] = (w.m0 + r < M && k0 + kq + i < K) ? w.A[static_cast<int64_t>(w.m0 + r) * lda + k0 + kq + i] : 0.0f;
                    }
                }
                else
                {
                    const int kk = tid >> 4, mq = (tid & 15) * 4; // A[k0 + kk][m0 + mq ..]
                    if (WHOLE || (vec_a && k0 + kk < K && w.m0 + mq + 3 < M))
                        v = *reinterpret_cast<const f4*>(w.A + static_cast<int64_t>(k0 + kk) * lda + w.m0 + mq);
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[i] = (k0 + kk < K && w.m0 + mq + i < M) ? w.A[static_cast<int64_t>(k0 + kk) * lda + w.m0 + mq + i] : 0.0f;
                    }
                }
                return v;
            };
            auto put_a = [&](f4 v, int kbase) {
                if (!ta)
                {
                    const int r = tid >> 2, kq = (tid & 3) * 4;
                    *reinterpret_cast<f4*>(&as[a_at(kbase + kq, r)]) = v;
                }
                else
                {
                    const int kk = tid >> 4, mq = (tid & 15) * 4;
                    *reinterpret_cast<f4*>(&as[a_at(kbase + kk, mq)]) = v;
                }
            };
            auto fetch_b = [&](const TileAt& w, int k0) -> f4 {
                f4 v = f4{0.0f, 0.0f, 0.0f, 0.0f};
                if (!tb)
                {
                    const int kk = tid >> 4, nq = (tid & 15) * 4; // B[k0 + kk][n0 + nq ..]
                    if (WHOLE || (vec_b && k0 + kk < K && w.n0 + nq + 3 < N))
                        v = *reinterpret_cast<const f4*>(w.B + static_cast<int64_t>(k0 + kk) * ldb + w.n0 + nq);
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[i] = (k0 + kk < K && w.n0 + nq + i < N) ? w.B[static_cast<int64_t>(k0 + kk) * ldb + w.n0 + nq + i] : 0.0f;
                    }
                }
                else
                {
                    const int r = tid >> 2, kq = (tid & 3) * 4; // B[n0 + r][k0 + kq ..]
                    if (WHOLE || (vec_b && w.n0 + r < N && k0 + kq + 3 < K))
                        v = *reinterpret_cast<const f4*>(w.B + static_cast<int64_t>(w.n0 + r) * ldb + k0 + kq);
                    else
                    {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            v[i] = (w.n0 + r < N && k0 + kq + i < K) ? w.B[static_cast<int64_t>(w.n0 + r) * ldb + k0 + kq + i] : 0.0f;
                    }
                }
                return v;
            };
            auto put_b = [&](f4 v, int kbase) {
                if (!tb)
                {
                    const int kk = tid >> 4, nq = (tid & 15) * 4;
                    *reinterpret_cast<f4*>(&bs[b_at(kbase + kk, nq)]) = v;
                }
                else
                {
                    const int r = tid >> 2, kq = (tid & 3) * 4;
                    *reinterpret_cast<f4*>(&bs[b_at(kbase + kq, r)]) = v;
                }
            };
            // (the optional quantized copy: Quantize of the f32 result, the arithmetic of hipq_quantize)
            const float qs = mq.out ? *mq.scale : 1.0f;
            const int32_t qz = mq.out ? load_zp(mq.zero_point, mq.quant_t) : 0;
            auto q1 = [&](float v) -> uint32_t {
                return mq.quant_t == HIPQ_U8 ? static_cast<uint32_t>(quantize_one<float, uint8_t>(v, qs, static_cast<uint8_t>(qz), mq.mode))
                                             : static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, int8_t>(v, qs, static_cast<int8_t>(qz), mq.mode)));
            };
            d4 acc[2][2];
            auto clear = [&]() {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
            };
            // block (i, j), register e of lane (r16, kq): row wm + 16 i + 4 e + kq, column wn + 16 j + r16.
            // A finished tile is rounded to f32 into `res` and stored one stage later, after the next
            // tile's operands have arrived: loads and stores share one counter, so stores issued just
            // before that wait would have to be acknowledged before the next tile could start.
            float res[2][2][4];
            auto round_tile = [&]() {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            res[i][j][e] = static_cast<float>(acc[i][j][e]);
            };
            auto each_result = [&](const TileAt& w, auto&& f) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                    {
                        const int m = w.m0 + wm + i * 16 + 4 * e + kq;
                        if (!WHOLE && m >= M)
                            continue;
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                        {
                            const int n = w.n0 + wn + j * 16 + r16;
                            if (!WHOLE && n >= N)
                                continue;
                            f(w.o_base + static_cast<int64_t>(m) * ldo + n, res[i][j][e]);
                        }
                    }
            };
            auto store_tile = [&](const TileAt& w) {
                if (out) // uniform
                    each_result(w, [&](int64_t at, float r) { out[at] = r; });
                if (mq.out) // uniform
                    each_result(w, [&](int64_t at, float r) { static_cast<uint8_t*>(mq.out)[at] = static_cast<uint8_t>(q1(r)); });
            };

            if (item >= tiles) // uniform
                return;
            // a stage is TK of the reduction (the whole reduction of an attention score), asked for at once
            constexpr int PIECES = TK / TKS;
            int t_fetch = item, k_fetch = 0, k_done = 0;
            TileAt ft = tile_at(t_fetch); // the tile whose operands are being fetched
            TileAt ct = ft;               // the tile being multiplied
            TileAt st = ft;               // the finished tile waiting in `res`
            bool unsaved = false;         // uniform
            f4 va[PIECES], vb[PIECES];
#pragma unroll
            for (int q = 0; q < PIECES; ++q)
            {
                va[q] = fetch_a(ft, q * TKS);
                vb[q] = fetch_b(ft, q * TKS);
            }
            clear();
            for (;;)
            {
#pragma unroll
                for (int q = 0; q < PIECES; ++q)
                {
                    put_a(va[q], q * TKS);
                    put_b(vb[q], q * TKS);
                }
                __syncthreads();
                // the stage after this one: of this tile, or the first of the workgroup's next tile
                bool more = true; // uniform
                k_fetch += TK;
                if (k_fetch >= K)
                {
                    k_fetch = 0;
                    t_fetch += grid;
                    more = t_fetch < tiles;
                    if (more)
                        ft = tile_at(t_fetch);
                }
                if (more)
                {
#pragma unroll
                    for (int q = 0; q < PIECES; ++q)
                    {
                        va[q] = fetch_a(ft, k_fetch + q * TKS);
                        vb[q] = fetch_b(ft, k_fetch + q * TKS);
                    }
                }
                if (unsaved)
                {
                    store_tile(st);
                    unsaved = false;
                }
#pragma unroll
                for (int k = 0; k < TK; k += 4)
                {
                    // (past K both operands hold zeros: + 0 * 0 leaves a sum as it is -- a sum that started from +0 is never -0)
                    double ad[2], bd[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                    {
                        ad[i] = static_cast<double>(as[a_at(k + kq, wm + i * 16 + r16)]);
                        bd[i] = static_cast<double>(bs[b_at(k + kq, wn + i * 16 + r16)]);
                    }
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ad[i], bd[j], acc[i][j], 0, 0, 0);
                }
                __syncthreads();
                k_done += TK;
                if (k_done >= K) // the tile's last stage: the fetch cursor stands on the next tile
                {
                    round_tile();
                    st = ct;
                    if (!more)
                        break;
                    unsaved = true;
                    clear();
                    k_done = 0;
                    ct = ft;
                }
            }
            store_tile(st);
        }

        // ---- attention of one head in one kernel -------------------------------------------------------
        // out = BatchMatMul(Softmax(Multiply(BatchMatMulTranspose(Q, K), factor)), V), every op rounding
        // as the separate kernels round (the products through the same matrix instruction chain, the
        // Softmax with the same lanes on the same elements as the Softmax kernel of that row length), so
        // the result equals the three launches bit for bit while the scores never leave the compute unit.
        // A workgroup takes RB blocks of 16 query rows of one head against all of its keys, depth 64.  Keys
        // and values pass through one LDS region in chunks of 128 (those beyond the last key are neither
        // multiplied nor summed), the next chunk on its way into registers while one is multiplied; every
        // wavefront keeps the fragments of Q, which pass through the region that then holds the scores.
        // Rows of Q, K and the scores are four floats longer than their data, so that fragment reads (16 rows
        // x 4 consecutive k a wavefront) and the 16-byte writes touch every bank once at offsets known at
        // compile time; rows of V are swizzled by n ^ 16 (key % 4).  32 rows x 384 keys are swizzled by
        // column ^ 4 (row % 16) instead: without the four floats two workgroups fit a compute unit's LDS,
        // and one multiplies while the other waits at a barrier or exponentiates (1440 items of 32 x 384:
        // 112 us, with one workgroup a compute unit 133; the three launches 120).
        // Bound by the f64 matrix instruction (64 cycles each) plus, not beside, the vector work of a SIMD:
        // at 384 heads of 128 x 128 the instruction alone takes 20 us, the kernel 39 (with the swizzle
        // computed for every fragment 42, as a resident grid that walks the items 42); 12 heads: 6.5 us
        // (8 wavefronts on 32 rows 9.3; the three launches 18.5).
        constexpr int AKEYS = 128, AD = 64; // keys of a chunk, depth
        constexpr int AMAX = 512;          // keys
        struct AttnView
        {
            int64_t batch_inner;
            int64_t q_outer, q_inner, ldq;
            int64_t k_outer, k_inner, ldk;
            int64_t v_outer, v_inner, ldv;
            int64_t o_outer, o_inner, ldo;
        };
        // floats a row of Q, K and the scores is longer than its data; none: swizzled instead
        constexpr int attn_pad(int rb, int chunks) { return rb == 2 && chunks == 3 ? 0 : 4; }
        constexpr size_t attn_lds(int rb, int chunks)
        {
            return (static_cast<size_t>(rb) * 16 * (AKEYS * chunks + attn_pad(rb, chunks)) + AKEYS * (AD + attn_pad(rb, chunks))) * sizeof(float);
        }

        // CH: chunks of keys; WHOLE: the keys fill them (a number known at compile time, and nothing to check)
        template <int RB, int WAVES, int CH, bool WHOLE>
        __global__ __launch_bounds__(WAVES * 64, 4) void attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                                                              const float* __restrict__ factor, float* __restrict__ out, AttnView view, MatQuant mq, int32_t queries,
                                                                              int32_t keys_, int32_t row_blocks)
        {
            touch_arguments<40 + sizeof(AttnView) + sizeof(MatQuant)>();
            const int keys = WHOLE ? CH * AKEYS : keys_;
            constexpr int QB = RB * 16;
            constexpr int ROWS = WAVES * 4;      // rows that one piece a thread covers
            constexpr int PIECES = AKEYS / ROWS; // 16-byte pieces a thread and chunk
            constexpr int KB = 8 / WAVES;                            // 16-key blocks of a chunk a wavefront multiplies
            constexpr int CB = RB * 4 >= WAVES ? RB * 4 / WAVES : 1; // 16 x 16 blocks of the context a wavefront owns
            constexpr int PAD = attn_pad(RB, CH);
            constexpr int pitch = CH * AKEYS + PAD, kpitch = AD + PAD; // of a row of scores, of a row of Q and K
            static_assert(QB <= ROWS, "a piece of Q a thread");
            extern __shared__ __attribute__((aligned(16))) float attn_lds_base[];
            float* const Ss = attn_lds_base;
            float* const KV = Ss + QB * pitch;
            const int tid = threadIdx.x;
            const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int r16 = lane & 15, kq = lane >> 4;
            const int64_t ldq = view.ldq, ldk = view.ldk, ldv = view.ldv, ldo = view.ldo;
            const bool scaled = factor != nullptr;
            const float c = scaled ? *factor : 1.0f;
            const int grid = static_cast<int>(gridDim.x);
            // (workgroups are dealt round-robin to the 8 XCDs: renumbered so that the row blocks of a head meet in one L2)
            const int t = (grid & 7) == 0 ? (static_cast<int>(blockIdx.x) & 7) * (grid >> 3) + (static_cast<int>(blockIdx.x) >> 3) : static_cast<int>(blockIdx.x);
            const int rb = t % row_blocks;
            const uint32_t batch = static_cast<uint32_t>(t / row_blocks);
            const uint32_t batch_inner = static_cast<uint32_t>(view.batch_inner < (1ll << 31) ? view.batch_inner : (1ll << 31));
            const int64_t bo = batch / batch_inner, bi = batch - bo * batch_inner;
            const float* const Q = q + bo * view.q_outer + bi * view.q_inner + static_cast<int64_t>(rb) * QB * ldq;
            const float* const K = k + bo * view.k_outer + bi * view.k_inner;
            const float* const V = v + bo * view.v_outer + bi * view.v_inner;
            const int64_t o_base = bo * view.o_outer + bi * view.o_inner + static_cast<int64_t>(rb) * QB * ldo;
            const int rows = min(QB, queries - rb * QB); // query rows that exist
            // a thread's 16-byte pieces: row tid / 16 (+ ROWS a piece), columns 4 (tid % 16) ..
            const int prow = tid >> 4, pcol = (tid & 15) * 4;
            // (the compiler would compute every address of the loops below once and keep it: hundreds of registers.
            // A value that it cannot see through makes it form them where they are used)
            auto fresh = [](int x) {
                asm volatile("" : "+v"(x));
                return x;
            };
            f4 rkv[PIECES];
            auto fetch = [&](const float* from, int64_t ld, int chunk) {
                const int row0 = chunk * AKEYS + fresh(tid >> 4);
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
                {
                    const int row = WHOLE ? row0 + ROWS * i : min(row0 + ROWS * i, keys - 1); // (keys past the last are not scored)
                    rkv[i] = *reinterpret_cast<const f4*>(from + static_cast<int64_t>(row) * ld + pcol);
                }
            };
            auto swizzled = [](int col, int row) { return PAD ? col : col ^ (4 * (row & 15)); };
            auto put_k = [&]() {
                const int at = prow * kpitch + swizzled(pcol, prow); // (row % 16 = (tid / 16) % 16 for every piece of the thread)
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
                    *reinterpret_cast<f4*>(KV + at + i * ROWS * kpitch) = rkv[i];
            };
            auto put_v = [&](int chunk) {
                const int at = prow * AD + (pcol ^ (16 * (prow & 3))); // (key % 4 = (tid / 16) % 4 for every piece)
#pragma unroll
                for (int i = 0; i < PIECES; ++i)
                {
                    // (values past the last key meet zero probabilities: zeros themselves, whatever the last row holds)
                    const f4 zero = f4{0.0f, 0.0f, 0.0f, 0.0f};
                    *reinterpret_cast<f4*>(KV + at + i * ROWS * AD) = (WHOLE || chunk * AKEYS + prow + ROWS * i < keys) ? rkv[i] : zero;
                }
            };
            {
                const f4 piece = *reinterpret_cast<const f4*>(Q + static_cast<int64_t>(min(prow, rows - 1)) * ldq + pcol); // (rows past the last are not stored)
                fetch(K, ldk, 0);
                if (QB == ROWS || prow < QB)
                    *reinterpret_cast<f4*>(Ss + prow * kpitch + swizzled(pcol, prow)) = piece;
                put_k();
            }
            // ---- scores, a chunk of keys at a time; this wavefront KB blocks of 16 keys of every chunk
            float qf[RB][AD / 4];
#pragma unroll
            for (int ch = 0; ch < CH; ++ch)
            {
                __syncthreads(); // the chunk (and Q) is in LDS
                if (ch + 1 < CH)
                    fetch(K, ldk, ch + 1);
                else
                    fetch(V, ldv, 0);
                const int swz = PAD ? 0 : fresh(4 * r16);
                if (ch == 0)
                {
#pragma unroll
                    for (int s = 0; s < AD / 4; ++s)
#pragma unroll
                        for (int i = 0; i < RB; ++i)
                            qf[i][s] = Ss[(16 * i + r16) * kpitch + ((4 * s) ^ swz) + kq];
                }
                const int key0 = ch * AKEYS + wave * KB * 16;
                d4 acc[RB][KB];
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < KB; ++j)
                        acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
                const bool some = WHOLE || ch + 1 < CH || key0 < keys; // uniform
                if (some)
                {
                    const float* const kb = KV + (wave * KB * 16 + r16) * kpitch + kq;
#pragma unroll
                    for (int s = 0; s < AD / 4; ++s)
                    {
                        double bd[KB];
#pragma unroll
                        for (int j = 0; j < KB; ++j)
                            bd[j] = static_cast<double>(kb[((4 * s) ^ swz) + j * 16 * kpitch]);
#pragma unroll
                        for (int i = 0; i < RB; ++i)
#pragma unroll
                            for (int j = 0; j < KB; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(qf[i][s]), bd[j], acc[i][j], 0, 0, 0);
                    }
                }
                __syncthreads(); // every wavefront has read the chunk (and Q): the next one takes its place
                if (some)
                {
#pragma unroll
                    for (int i = 0; i < RB; ++i)
#pragma unroll
                        for (int j = 0; j < KB; ++j)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                            {
                                const int row = 4 * e + kq;
                                Ss[(16 * i + row) * pitch + swizzled(key0 + 16 * j + r16, row)] = static_cast<float>(acc[i][j][e]);
                            }
                }
                if (ch + 1 < CH)
                    put_k();
                else
                    put_v(0);
            }
            __syncthreads();
            // ---- Softmax: 32 lanes a row as in the Softmax kernel, two rows a wavefront at a time
#pragma unroll
            for (int it = 0; it < QB / WAVES / 2; ++it)
            {
                const int row = QB / WAVES * wave + 2 * it + (lane >> 5);
                f4* const at = reinterpret_cast<f4*>(Ss + row * pitch + swizzled(4 * (lane & 31), row));
                f4 p[CH];
#pragma unroll
                for (int i = 0; i < CH; ++i)
                    p[i] = at[32 * i];
                softmax_row<32, CH>(p, lane & 31, keys, scaled, c);
#pragma unroll
                for (int i = 0; i < CH; ++i)
                    at[32 * i] = p[i]; // (zeros past the last key)
            }
            // ---- context over the keys, a chunk at a time: this wavefront's blocks are row blocks cr .. cr + CB - 1
            // of column block cc; register e of lane (r16, kq) is row 4 e + kq, column r16 of a block
            const int cc = wave & 3;
            const int cr = WAVES == 4 ? 0 : (wave >> 2) * CB;
            const bool has_context = RB * 4 >= WAVES || wave < RB * 4; // uniform
            d4 ctx[CB];
#pragma unroll
            for (int i = 0; i < CB; ++i)
                ctx[i] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int ch = 0; ch < CH; ++ch)
            {
                __syncthreads(); // the chunk of V (and the probabilities) are in LDS
                if (ch + 1 < CH)
                    fetch(V, ldv, ch + 1);
                if (has_context)
                {
                    const int swz = PAD ? 0 : fresh(4 * r16);
                    const float* const pa = Ss + (cr * 16 + r16) * pitch + kq + ch * AKEYS;
                    const float* const vb = KV + kq * AD + ((16 * cc + r16) ^ (16 * kq));
#pragma unroll
                    for (int g = 0; g < AKEYS / 16; ++g)
                        if (WHOLE || ch + 1 < CH || ch * AKEYS + g * 16 < keys) // uniform
                        {
#pragma unroll
                            for (int s = 4 * g; s < 4 * g + 4; ++s)
                            {
                                const double bd = static_cast<double>(vb[4 * s * AD]);
#pragma unroll
                                for (int i = 0; i < CB; ++i)
                                    ctx[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(pa[((4 * s) ^ swz) + i * 16 * pitch]), bd, ctx[i], 0, 0, 0);
                            }
                        }
                }
                if (ch + 1 < CH)
                {
                    __syncthreads(); // every wavefront has read the chunk
                    put_v(ch + 1);
                }
            }
            if (!has_context)
                return;
            const float qs = mq.out ? *mq.scale : 1.0f;
            const int32_t qz = mq.out ? load_zp(mq.zero_point, mq.quant_t) : 0;
            const bool rne = mq.mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN; // uniform: the Quantize kernels' four-at-a-time arithmetic
#pragma unroll
            for (int i = 0; i < CB; ++i)
            {
                const f4 x = f4{static_cast<float>(ctx[i][0]), static_cast<float>(ctx[i][1]), static_cast<float>(ctx[i][2]), static_cast<float>(ctx[i][3])};
                uint32_t four = 0;
                if (mq.out && rne)
                    four = mq.quant_t == HIPQ_U8 ? quantize4<uint8_t, true>(x, qs, static_cast<float>(qz), mq.mode) : quantize4<int8_t, true>(x, qs, static_cast<float>(qz), mq.mode);
                else if (mq.out)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        four |= (mq.quant_t == HIPQ_U8 ? static_cast<uint32_t>(quantize_one<float, uint8_t>(x[e], qs, static_cast<uint8_t>(qz), mq.mode))
                                                       : static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, int8_t>(x[e], qs, static_cast<int8_t>(qz), mq.mode))))
                                << (8 * e);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const int row = 16 * (cr + i) + 4 * e + kq;
                    if (row >= rows)
                        continue;
                    const int64_t at = o_base + static_cast<int64_t>(row) * ldo + 16 * cc + r16;
                    if (out) // uniform
                        out[at] = x[e];
                    if (mq.out) // uniform
                        static_cast<uint8_t*>(mq.out)[at] = static_cast<uint8_t>(four >> (8 * e));
                }
            }
        }

        template <int RB, int WAVES>
        int launch_attention(const float* q, const float* k, const float* v, const float* factor, float* out, const AttnView& av, const MatQuant& mq, int64_t batch, int64_t queries, int64_t keys,
                             hipStream_t s)
        {
            const int ch = static_cast<int>((keys + AKEYS - 1) / AKEYS);
            const auto kernel = keys == AKEYS ? attention_f32_kernel<RB, WAVES, 1, true>
                                : ch == 1     ? attention_f32_kernel<RB, WAVES, 1, false>
                                : ch == 2     ? attention_f32_kernel<RB, WAVES, 2, false>
                                : ch == 3     ? attention_f32_kernel<RB, WAVES, 3, false>
                                              : attention_f32_kernel<RB, WAVES, 4, false>;
            static bool configured[16][5] = {};
            const int which = keys == AKEYS ? 0 : ch;
            int dev = 0;
            HIPQ_HIP(hipGetDevice(&dev));
            if (dev >= 0 && dev < 16 && !configured[dev][which])
            {
                HIPQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
                configured[dev][which] = true;
            }
            const int64_t row_blocks = (queries + RB * 16 - 1) / (RB * 16);
            HIPQ_REQUIRE(batch * row_blocks < (1ll << 31) - (1 << 20), "too many work items for one launch");
            kernel<<<static_cast<unsigned>(batch * row_blocks), WAVES * 64, attn_lds(RB, ch), s>>>(q, k, v, factor, out, av, mq, static_cast<int32_t>(queries), static_cast<int32_t>(keys),
                                                                                                    static_cast<int32_t>(row_blocks));
            return check_launch("attention_f32");
        }
    }
}

using namespace hipq;

static int launch_batch_matmul(const float* a, const float* b, float* out, const MatView& view, const MatQuant& mq, int64_t batch, int64_t M, int64_t K, int64_t N, int32_t transpose_a,
                               int32_t transpose_b, void* stream)
{
    HIPQ_REQUIRE(M < (1ll << 31) && K < (1ll << 31) && N < (1ll << 31), "extent too large");
    const int64_t m_tiles = (M + TM - 1) / TM, n_tiles = (N + TN - 1) / TN;
    // 16-byte accesses along the rows when every row of every matrix starts aligned
    auto all4 = [](int64_t x, int64_t y, int64_t z) { return x % 4 == 0 && y % 4 == 0 && z % 4 == 0; };
    const int vec_a = (reinterpret_cast<uintptr_t>(a) & 15) == 0 && all4(view.lda, view.a_outer, view.a_inner);
    const int vec_b = (reinterpret_cast<uintptr_t>(b) & 15) == 0 && all4(view.ldb, view.b_outer, view.b_inner);
    HIPQ_REQUIRE(batch * m_tiles * n_tiles < (1ll << 31) - (1 << 20), "too many tiles for one launch");
    const int64_t tiles = batch * m_tiles * n_tiles;
    // three workgroups a compute unit (their LDS and the 12 wavefronts they make fit), each walking its share of the tiles
    const int64_t grid = std::min<int64_t>(tiles, static_cast<int64_t>(BMM_PER_CU) * device_compute_units());
    const bool whole = M % TM == 0 && N % TN == 0 && K % TK == 0 && K > 0 && vec_a && vec_b;
#define BMM_LAUNCH(W, TA, TB)                                                                                                                                                            \
    batch_matmul_f32_kernel<W, TA, TB><<<static_cast<unsigned>(grid), 256, 0, as_stream(stream)>>>(a, b, out, view, mq, static_cast<int32_t>(M), static_cast<int32_t>(K), static_cast<int32_t>(N), \
                                                                                                     static_cast<int32_t>(m_tiles), static_cast<int32_t>(n_tiles), static_cast<int32_t>(tiles), vec_a, vec_b)
#define BMM_T(W) (transpose_a ? (transpose_b ? BMM_LAUNCH(W, true, true) : BMM_LAUNCH(W, true, false)) : (transpose_b ? BMM_LAUNCH(W, false, true) : BMM_LAUNCH(W, false, false)))
    if (whole)
        BMM_T(true);
    else
        BMM_T(false);
#undef BMM_T
#undef BMM_LAUNCH
    return check_launch("batch_matmul_f32");
}

int hipq_batch_matmul_f32(const float* a, const float* b, float* out, int64_t batch, int64_t M, int64_t K, int64_t N, int32_t transpose_a, int32_t transpose_b, void* stream)
{
    HIPQ_REQUIRE(batch >= 0 && M >= 0 && K >= 0 && N >= 0, "negative extent");
    if (batch == 0 || M == 0 || N == 0)
        return HIPQ_OK;
    HIPQ_REQUIRE(out && (K == 0 || (a && b)), "null pointer");
    HIPQ_REQUIRE((reinterpret_cast<uintptr_t>(out) & 15) == 0, "the output must be 16-byte aligned");
    const MatView view{1, M * K, 0, transpose_a ? M : K, K * N, 0, transpose_b ? K : N, M * N, 0, N};
    return launch_batch_matmul(a, b, out, view, MatQuant{nullptr, nullptr, nullptr, HIPQ_I8, HIPQ_ROUND_NEAREST_TOWARD_EVEN}, batch, M, K, N, transpose_a, transpose_b, stream);
}

int hipq_batch_matmul_view_f32(const float* a, const float* b, float* out, const hipq_matmul_view_t* v, const hipq_quant_out_t* q, int64_t batch, int64_t M, int64_t K, int64_t N,
                               int32_t transpose_a, int32_t transpose_b, void* stream)
{
    HIPQ_REQUIRE(v, "null view");
    HIPQ_REQUIRE(batch >= 0 && M >= 0 && K >= 0 && N >= 0, "negative extent");
    if (batch == 0 || M == 0 || N == 0)
        return HIPQ_OK;
    MatQuant mq{nullptr, nullptr, nullptr, HIPQ_I8, HIPQ_ROUND_NEAREST_TOWARD_EVEN};
    if (q)
    {
        HIPQ_REQUIRE(q->out && q->scale, "quantized output: null pointer");
        HIPQ_REQUIRE(q->quant_t == HIPQ_I8 || q->quant_t == HIPQ_U8, "quantized output: i8 or u8");
        HIPQ_REQUIRE(q->round_mode >= HIPQ_ROUND_NEAREST_TOWARD_INFINITY && q->round_mode <= HIPQ_ROUND_DOWN, "quantized output: unknown round mode");
        mq = MatQuant{q->out, q->scale, q->zero_point, q->quant_t, q->round_mode};
    }
    HIPQ_REQUIRE((out || mq.out) && (K == 0 || (a && b)), "null pointer");
    HIPQ_REQUIRE(v->batch_inner >= 1, "batch_inner must be at least 1");
    HIPQ_REQUIRE(v->lda >= (transpose_a ? M : K) && v->ldb >= (transpose_b ? K : N) && v->ldo >= N, "a row stride is shorter than the row");
    HIPQ_REQUIRE(v->a_outer >= 0 && v->a_inner >= 0 && v->b_outer >= 0 && v->b_inner >= 0 && v->o_outer >= 0 && v->o_inner >= 0, "negative batch stride");
    const MatView view{v->batch_inner, v->a_outer, v->a_inner, v->lda, v->b_outer, v->b_inner, v->ldb, v->o_outer, v->o_inner, v->ldo};
    return launch_batch_matmul(a, b, out, view, mq, batch, M, K, N, transpose_a, transpose_b, stream);
}

int hipq_attention_f32(const float* q, const float* k, const float* v, const float* factor, float* out, const hipq_attention_view_t* view, const hipq_quant_out_t* quant, int64_t batch,
                       int64_t queries, int64_t keys, int64_t depth, void* stream)
{
    HIPQ_REQUIRE(view, "null view");
    HIPQ_REQUIRE(batch >= 0 && queries >= 0 && keys >= 0 && depth >= 0, "negative extent");
    // (every length up to the largest: 17 x 17 12 heads 6.0 us here and 17.6 in three launches, 64 x 64, a whole tile of
    // the products' own kernel, 6.2 and 15.8, 768 heads 28.3 and 35.4, 65 x 65 48.7 and 96.6)
    const bool self = queries == keys && keys > 0 && keys <= AMAX;
    if (depth != AD || !(self || (keys == AKEYS && queries % 32 == 0)))
        return fail(HIPQ_ERR_UNSUPPORTED, "the one-kernel attention takes depth 64 and as many queries as keys, up to 512, or 128 keys and query rows in multiples of 32 (run the three ops otherwise)");
    if (batch == 0 || queries == 0)
        return HIPQ_OK;
    MatQuant mq{nullptr, nullptr, nullptr, HIPQ_I8, HIPQ_ROUND_NEAREST_TOWARD_EVEN};
    if (quant)
    {
        HIPQ_REQUIRE(quant->out && quant->scale, "quantized output: null pointer");
        HIPQ_REQUIRE(quant->quant_t == HIPQ_I8 || quant->quant_t == HIPQ_U8, "quantized output: i8 or u8");
        HIPQ_REQUIRE(quant->round_mode >= HIPQ_ROUND_NEAREST_TOWARD_INFINITY && quant->round_mode <= HIPQ_ROUND_DOWN, "quantized output: unknown round mode");
        mq = MatQuant{quant->out, quant->scale, quant->zero_point, quant->quant_t, quant->round_mode};
    }
    HIPQ_REQUIRE(q && k && v && (out || mq.out), "null pointer");
    HIPQ_REQUIRE(view->batch_inner >= 1, "batch_inner must be at least 1");
    HIPQ_REQUIRE(view->ldq >= depth && view->ldk >= depth && view->ldv >= depth && view->ldo >= depth, "a row stride is shorter than the row");
    HIPQ_REQUIRE(view->q_outer >= 0 && view->q_inner >= 0 && view->k_outer >= 0 && view->k_inner >= 0 && view->v_outer >= 0 && view->v_inner >= 0 && view->o_outer >= 0 && view->o_inner >= 0,
                 "negative batch stride");
    auto rows16 = [](const float* p, int64_t ld, int64_t outer, int64_t inner) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 4 == 0 && outer % 4 == 0 && inner % 4 == 0; };
    HIPQ_REQUIRE(rows16(q, view->ldq, view->q_outer, view->q_inner) && rows16(k, view->ldk, view->k_outer, view->k_inner) && rows16(v, view->ldv, view->v_outer, view->v_inner),
                 "rows of Q, K and V must start 16-byte aligned");
    const AttnView av{view->batch_inner, view->q_outer, view->q_inner, view->ldq, view->k_outer, view->k_inner, view->ldk,
                      view->v_outer, view->v_inner, view->ldv, view->o_outer, view->o_inner, view->ldo};
    // 16 query rows a workgroup, or 32: two blocks of rows share the fragments of K, the chunks staged and the
    // barriers, so that an item of 32 rows costs about 1.75 items of 16, measured from 12 x 128 x 128 to 120 x
    // 384 x 384; whichever leaves the fullest compute unit with less
    const int64_t cus = device_compute_units();
    auto items_a_cu = [&](int64_t rows) { return (batch * ((queries + rows - 1) / rows) + cus - 1) / cus; };
    if (4 * items_a_cu(16) <= 7 * items_a_cu(32))
        return launch_attention<1, 8>(q, k, v, factor, out, av, mq, batch, queries, keys, as_stream(stream));
    return launch_attention<2, 8>(q, k, v, factor, out, av, mq, batch, queries, keys, as_stream(stream));
}
