// Quantize / Dequantize kernels (HBM-bound elementwise work).
//
// Arithmetic follows src/ngraph/runtime/reference/quantize.hpp:29-117 and dequantize.hpp:31-53 of
// the nGraph tree: true IEEE division by the scale, the reference's floor/ceil rounding formulas,
// zero point added in REAL, clamp in REAL, then the cast.
//
// Three kernel families:
//   *_vec4    f32 <-> {i8,u8}, scale laid along one run of adjacent axes (or scalar) and the
//             innermost non-axis extent a multiple of 4.  Each lane moves groups of 4 elements:
//             one 16-byte load/store on the f32 side, one 4-byte store/load on the quantized side,
//             lane-contiguous, so a wavefront touches 1 KiB + 256 B of consecutive memory per step.
//   *_ragged  the same types and the same accesses where a group of 4 may reach into the next row of
//             the scale table (an inner extent that is no multiple of 4) or past the end.
//   *_generic every other case (f64, i32, scattered axes): one element per lane, coordinates
//             recovered with 64-bit div/mod.
#include "hipq_common.h"
#include "hipq_index_div.h"
#include "hipq_quant_math.h"

namespace hipq
{
    struct DimInfo
    {
        int32_t rank;
        uint32_t axes_mask;
        int64_t shape[HIPQ_MAX_RANK];
    };

    __device__ __forceinline__ int64_t project_index(const DimInfo& d, int64_t i)
    {
        int64_t coord[HIPQ_MAX_RANK];
        for (int a = d.rank - 1; a >= 0; --a)
        {
            coord[a] = i % d.shape[a];
            i /= d.shape[a];
        }
        int64_t j = 0;
        for (int a = 0; a < d.rank; ++a)
            if (d.axes_mask & (1u << a))
                j = j * d.shape[a] + coord[a];
        return j;
    }

    template <typename REAL, typename QUANT>
    __global__ __launch_bounds__(256) void quantize_generic_kernel(const REAL* __restrict__ in,
                                                                   const REAL* __restrict__ scale,
                                                                   const QUANT* __restrict__ zp,
                                                                   QUANT* __restrict__ out,
                                                                   int64_t count,
                                                                   DimInfo dims,
                                                                   int mode)
    {
        int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
        for (; i < count; i += stride)
        {
            int64_t j = dims.axes_mask ? project_index(dims, i) : 0;
            out[i] = quantize_one<REAL, QUANT>(in[i], scale[j], zp[j], mode);
        }
    }

    template <typename QUANT, typename REAL>
    __global__ __launch_bounds__(256) void dequantize_generic_kernel(const QUANT* __restrict__ in,
                                                                     const REAL* __restrict__ scale,
                                                                     const QUANT* __restrict__ zp,
                                                                     REAL* __restrict__ out,
                                                                     int64_t count,
                                                                     DimInfo dims)
    {
        int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
        for (; i < count; i += stride)
        {
            int64_t j = dims.axes_mask ? project_index(dims, i) : 0;
            // integer subtract after promotion; int32 wraps (dequantize.hpp:46-50)
            int32_t diff = static_cast<int32_t>(static_cast<uint32_t>(static_cast<int32_t>(in[i])) -
                                                static_cast<uint32_t>(static_cast<int32_t>(zp[j])));
            out[i] = static_cast<REAL>(diff) * scale[j];
        }
    }

    // ---- vectorised f32 <-> 8-bit path ----------------------------------------------------------
    // The tensor is viewed as [outer, A, inner] with the scale index = (i / inner) % A
    // (A == 1: scalar scale).  groups = count / 4; group g covers elements 4g .. 4g+3.
    struct RunView
    {
        IndexDiv div_inner4; // divides a group index by inner/4
        IndexDiv div_a;
        uint32_t a;         // extent of the scale table
    };

    __device__ __forceinline__ uint32_t run_index(const RunView& v, uint32_t group)
    {
        if (v.a == 1)
            return 0;
        uint32_t row = fastdiv(group, v.div_inner4);
        uint32_t q = fastdiv(row, v.div_a);
        return row - q * v.a;
    }

    // Groups a lane handles per launch, one wavefront-contiguous step of 256 groups apart (measured
    // on f32[64,1024,1024]: 3 is best for Quantize, 2 for Dequantize).  A short tensor, whose steps do
    // not fill the compute units eight times, takes one: it waits for one load and not for bandwidth,
    // and shorter workgroups spread over more compute units (both directions of f32[13, 1, 16868]: 5.34
    // us with the long ones, 4.12 so).
    constexpr int kQuantUnroll = 3;
    constexpr int kDequantUnroll = 2;

    // ROW_UNIFORM: inner/4 is a multiple of the 256 groups one step of a workgroup covers (or the
    // scale is a scalar), so a step lies inside one row of the scale table and its index comes from
    // the block index alone: scale and zero point arrive through the scalar unit instead of two
    // vector loads and two 64-bit multiplies per lane.
    template <bool ROW_UNIFORM>
    __device__ __forceinline__ uint32_t step_run_index(const RunView& v, uint32_t first_group_of_step, uint32_t g)
    {
        return run_index(v, ROW_UNIFORM ? first_group_of_step : g);
    }
    template <typename QUANT, bool RNE, bool ROW_UNIFORM, int UNROLL>
    __global__ __launch_bounds__(256) void quantize_vec4_kernel(const f32x4* __restrict__ in,
                                                                const float* __restrict__ scale,
                                                                const QUANT* __restrict__ zp,
                                                                uint32_t* __restrict__ out,
                                                                uint32_t groups,
                                                                RunView view,
                                                                int mode)
    {
        uint32_t first = blockIdx.x * (256u * UNROLL);
        uint32_t base = first + threadIdx.x;
        f32x4 x[UNROLL];
        float s[UNROLL];
        float z[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            uint32_t g = base + u * 256u;
            if (g < groups)
            {
                x[u] = __builtin_nontemporal_load(&in[g]);
                uint32_t j = step_run_index<ROW_UNIFORM>(view, first + u * 256u, g);
                s[u] = scale[j];
                z[u] = static_cast<float>(zp[j]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            uint32_t g = base + u * 256u;
            if (g < groups)
                __builtin_nontemporal_store(quantize4<QUANT, RNE>(x[u], s[u], z[u], mode), &out[g]);
        }
    }

    // The quantized side is read with ordinary loads (4 bytes a lane: streaming hints on so narrow a
    // load cost a sixth of the rate), the f32 side written with streaming stores.
    template <typename QUANT, bool ROW_UNIFORM, int UNROLL>
    __global__ __launch_bounds__(256) void dequantize_vec4_kernel(const uint32_t* __restrict__ in,
                                                                  const float* __restrict__ scale,
                                                                  const QUANT* __restrict__ zp,
                                                                  f32x4* __restrict__ out,
                                                                  uint32_t groups,
                                                                  RunView view)
    {
        uint32_t first = blockIdx.x * (256u * UNROLL);
        uint32_t base = first + threadIdx.x;
        uint32_t q[UNROLL];
        float s[UNROLL];
        int32_t z[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            uint32_t g = base + u * 256u;
            if (g < groups)
            {
                q[u] = in[g];
                uint32_t j = step_run_index<ROW_UNIFORM>(view, first + u * 256u, g);
                s[u] = scale[j];
                z[u] = static_cast<int32_t>(zp[j]);
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            uint32_t g = base + u * 256u;
            if (g < groups)
            {
                float r[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    int32_t v = static_cast<int32_t>(static_cast<QUANT>((q[u] >> (8 * e)) & 0xFFu));
                    r[e] = __fmul_rn(static_cast<float>(v - z[u]), s[u]);
                }
                f32x4 o = {r[0], r[1], r[2], r[3]};
                __builtin_nontemporal_store(o, &out[g]);
            }
        }
    }

    // ---- rows of any length ----------------------------------------------------------------------
    // Groups of 4 consecutive elements whatever the rows' length: in a row of `inner` >= 4 a group lies in
    // one row or in two, and an element takes the parameters of the first as long as it is one of the
    // `left` that remain of it.  Bound by memory like the kernels above, and with their accesses (one
    // element a lane, its index by 64-bit division: f32[1, 894, 43045] 279 us for Quantize and Dequantize,
    // f32[1, 128, 51474] 57, f32[19, 834, 238] 35; so 75, 17 and 11.5).
    enum RaggedForm
    {
        RAGGED_STEP, // inner >= 1024: the 1024 elements of a workgroup's step lie in two rows at most, known from its index alone
        RAGGED_LANE, // inner >= 4: every lane looks its row up
        RAGGED_EACH  // shorter rows: every element does
    };
    struct RaggedView
    {
        IndexDiv div_inner, div_a;
        uint32_t inner, a, groups, tail; // full groups, elements behind the last
    };
    constexpr uint32_t kRaggedStep = 1024; // elements of a workgroup's step

    struct RaggedRow
    {
        uint32_t j0, j1; // scale index of the row that an element lies in, of the row behind it
        int32_t left;    // elements from this one to the row's end
    };
    __device__ __forceinline__ RaggedRow ragged_row(const RaggedView& v, uint32_t element)
    {
        const uint32_t row = fastdiv(element, v.div_inner);
        const uint32_t j = row - fastdiv(row, v.div_a) * v.a;
        return RaggedRow{j, j + 1 == v.a ? 0 : j + 1, static_cast<int32_t>((row + 1) * v.inner - element)};
    }

    template <typename QUANT, bool RNE, int FORM, int UNROLL>
    __global__ __launch_bounds__(256) void quantize_ragged_kernel(const float* __restrict__ in, const float* __restrict__ scale, const QUANT* __restrict__ zp, QUANT* __restrict__ out,
                                                                  RaggedView view, int mode)
    {
        const uint32_t first = blockIdx.x * (256u * UNROLL);
        f32x4 x[UNROLL];
        float s0[UNROLL], s1[UNROLL], z0[UNROLL], z1[UNROLL];
        int32_t left[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            const uint32_t step = first + u * 256u, g = step + threadIdx.x;
            if (FORM != RAGGED_EACH && g < view.groups)
            {
                x[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(in) + g);
                const RaggedRow r = ragged_row(view, 4 * (FORM == RAGGED_STEP ? step : g));
                s0[u] = scale[r.j0];
                s1[u] = scale[r.j1];
                z0[u] = static_cast<float>(zp[r.j0]);
                z1[u] = static_cast<float>(zp[r.j1]);
                left[u] = FORM == RAGGED_STEP ? r.left - 4 * static_cast<int32_t>(threadIdx.x) : r.left;
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            const uint32_t g = first + u * 256u + threadIdx.x;
            if (FORM != RAGGED_EACH && g < view.groups)
            {
                const bool in_first = left[u] > 0;
                uint32_t q = quantize4<QUANT, RNE>(x[u], in_first ? s0[u] : s1[u], in_first ? z0[u] : z1[u], mode);
                if (in_first && left[u] < 4)
                {
                    const uint32_t mask = (1u << (8 * left[u])) - 1;
                    q = (q & mask) | (quantize4<QUANT, RNE>(x[u], s1[u], z1[u], mode) & ~mask);
                }
                __builtin_nontemporal_store(q, reinterpret_cast<uint32_t*>(out) + g);
            }
            else if (FORM == RAGGED_EACH && g < view.groups)
            {
                const f32x4 v = reinterpret_cast<const f32x4*>(in)[g];
                uint32_t q = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const uint32_t j = ragged_row(view, 4 * g + e).j0;
                    q |= static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, QUANT>(v[e], scale[j], zp[j], RNE ? HIPQ_ROUND_NEAREST_TOWARD_EVEN : mode))) << (8 * e);
                }
                reinterpret_cast<uint32_t*>(out)[g] = q;
            }
            else if (g == view.groups)
            {
                for (uint32_t e = 0; e < view.tail; ++e)
                {
                    const uint32_t j = ragged_row(view, 4 * g + e).j0;
                    out[4 * g + e] = quantize_one<float, QUANT>(in[4 * g + e], scale[j], zp[j], mode);
                }
            }
        }
    }

    template <typename QUANT, int FORM, int UNROLL>
    __global__ __launch_bounds__(256) void dequantize_ragged_kernel(const QUANT* __restrict__ in, const float* __restrict__ scale, const QUANT* __restrict__ zp, float* __restrict__ out,
                                                                    RaggedView view)
    {
        const uint32_t first = blockIdx.x * (256u * UNROLL);
        uint32_t q[UNROLL];
        float s0[UNROLL], s1[UNROLL];
        int32_t z0[UNROLL], z1[UNROLL], left[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            const uint32_t step = first + u * 256u, g = step + threadIdx.x;
            if (FORM != RAGGED_EACH && g < view.groups)
            {
                q[u] = reinterpret_cast<const uint32_t*>(in)[g];
                const RaggedRow r = ragged_row(view, 4 * (FORM == RAGGED_STEP ? step : g));
                s0[u] = scale[r.j0];
                s1[u] = scale[r.j1];
                z0[u] = static_cast<int32_t>(zp[r.j0]);
                z1[u] = static_cast<int32_t>(zp[r.j1]);
                left[u] = FORM == RAGGED_STEP ? r.left - 4 * static_cast<int32_t>(threadIdx.x) : r.left;
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
        {
            const uint32_t g = first + u * 256u + threadIdx.x;
            if (FORM != RAGGED_EACH && g < view.groups)
            {
                f32x4 r;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const int32_t v = static_cast<int32_t>(static_cast<QUANT>((q[u] >> (8 * e)) & 0xFFu));
                    r[e] = __fmul_rn(static_cast<float>(v - (e < left[u] ? z0[u] : z1[u])), e < left[u] ? s0[u] : s1[u]);
                }
                __builtin_nontemporal_store(r, reinterpret_cast<f32x4*>(out) + g);
            }
            else if (FORM == RAGGED_EACH && g < view.groups)
            {
                const uint32_t b = reinterpret_cast<const uint32_t*>(in)[g];
                f32x4 r;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const uint32_t j = ragged_row(view, 4 * g + e).j0;
                    const int32_t v = static_cast<int32_t>(static_cast<QUANT>((b >> (8 * e)) & 0xFFu));
                    r[e] = __fmul_rn(static_cast<float>(v - static_cast<int32_t>(zp[j])), scale[j]);
                }
                reinterpret_cast<f32x4*>(out)[g] = r;
            }
            else if (g == view.groups)
            {
                for (uint32_t e = 0; e < view.tail; ++e)
                {
                    const uint32_t j = ragged_row(view, 4 * g + e).j0;
                    out[4 * g + e] = __fmul_rn(static_cast<float>(static_cast<int32_t>(in[4 * g + e]) - static_cast<int32_t>(zp[j])), scale[j]);
                }
            }
        }
    }

    // ---- host side -------------------------------------------------------------------------------
    struct Canon
    {
        int64_t count;
        bool single_run; // scalar, or one run of adjacent axes
        int64_t outer, a, inner;
    };

    static Canon canonicalise(const hipq_quant_desc_t& d)
    {
        Canon c;
        c.count = 1;
        for (int i = 0; i < d.rank; ++i)
            c.count *= d.shape[i];
        c.outer = c.a = c.inner = 1;
        // 0 = before the run, 1 = in the run, 2 = after the run
        int state = 0;
        c.single_run = true;
        for (int i = 0; i < d.rank; ++i)
        {
            if (d.shape[i] == 1)
                continue;
            bool on_axis = (d.axes_mask >> i) & 1u;
            if (on_axis)
            {
                if (state == 2)
                    c.single_run = false;
                state = 1;
                c.a *= d.shape[i];
            }
            else if (state == 0)
                c.outer *= d.shape[i];
            else
            {
                state = 2;
                c.inner *= d.shape[i];
            }
        }
        return c;
    }

    static int check_desc(const hipq_quant_desc_t* d)
    {
        HIPQ_REQUIRE(d, "descriptor is null");
        HIPQ_REQUIRE(d->rank >= 0 && d->rank <= HIPQ_MAX_RANK, "rank %d out of range", d->rank);
        for (int i = 0; i < d->rank; ++i)
            HIPQ_REQUIRE(d->shape[i] >= 0, "negative extent");
        HIPQ_REQUIRE((d->axes_mask >> d->rank) == 0, "axes beyond rank");
        if (d->real_t != HIPQ_F32 && d->real_t != HIPQ_F64)
            return fail(HIPQ_ERR_UNSUPPORTED, "real type must be f32 or f64");
        if (d->quant_t != HIPQ_U8 && d->quant_t != HIPQ_I8 && d->quant_t != HIPQ_I32)
            return fail(HIPQ_ERR_UNSUPPORTED, "quantized type must be u8, i8 or i32");
        return HIPQ_OK;
    }

    static DimInfo dim_info(const hipq_quant_desc_t& d)
    {
        DimInfo di;
        di.rank = d.rank;
        di.axes_mask = d.axes_mask;
        for (int i = 0; i < HIPQ_MAX_RANK; ++i)
            di.shape[i] = i < d.rank ? d.shape[i] : 1;
        return di;
    }

    static unsigned generic_blocks(int64_t count)
    {
        int64_t b = (count + 255) / 256;
        return static_cast<unsigned>(b > 65536 ? 65536 : (b < 1 ? 1 : b));
    }

    static bool ragged_ok(const hipq_quant_desc_t& d, const Canon& c, const void* f32_ptr, const void* q_ptr)
    {
        return d.real_t == HIPQ_F32 && (d.quant_t == HIPQ_U8 || d.quant_t == HIPQ_I8) && c.single_run && c.count < (1ll << 31) &&
               (reinterpret_cast<uintptr_t>(f32_ptr) & 15) == 0 && (reinterpret_cast<uintptr_t>(q_ptr) & 3) == 0;
    }
    // groups of 4 lie in one row of the scale table each
    static bool vec4_ok(const hipq_quant_desc_t& d, const Canon& c, const void* f32_ptr, const void* q_ptr)
    {
        return ragged_ok(d, c, f32_ptr, q_ptr) && c.count % 4 == 0 && (c.a == 1 || c.inner % 4 == 0);
    }

    // every 256-group step of a workgroup lies inside one row of the scale table
    static bool row_uniform(const Canon& c) { return c.a == 1 || (c.inner / 4) % 256 == 0; }

    static RunView make_view(const Canon& c)
    {
        RunView v;
        v.a = static_cast<uint32_t>(c.a);
        v.div_inner4 = make_fastdiv(static_cast<uint32_t>(c.a == 1 ? 1 : c.inner / 4));
        v.div_a = make_fastdiv(v.a);
        return v;
    }
    static RaggedView make_ragged_view(const Canon& c)
    {
        RaggedView v;
        v.a = static_cast<uint32_t>(c.a);
        v.inner = static_cast<uint32_t>(c.a == 1 ? c.count : c.inner);
        v.div_inner = make_fastdiv(v.inner);
        v.div_a = make_fastdiv(v.a);
        v.groups = static_cast<uint32_t>(c.count / 4);
        v.tail = static_cast<uint32_t>(c.count % 4);
        return v;
    }
    static RaggedForm ragged_form(const RaggedView& v) { return v.inner >= kRaggedStep ? RAGGED_STEP : (v.inner >= 4 ? RAGGED_LANE : RAGGED_EACH); }
    // (the group behind the last full one holds the tail)
    static unsigned ragged_blocks(const RaggedView& v, int unroll) { return (v.groups + 1 + 256 * unroll - 1) / (256 * unroll); }
    static bool is_short(uint32_t groups) { return (groups + 255) / 256 <= 8u * static_cast<unsigned>(device_compute_units()); }
}

using namespace hipq;

extern "C" {

int hipq_quantize(const hipq_quant_desc_t* d, const void* in, const void* scale, const void* zp, void* out, void* stream)
{
    int rc = check_desc(d);
    if (rc)
        return rc;
    HIPQ_REQUIRE(d->round_mode >= 0 && d->round_mode <= HIPQ_ROUND_DOWN, "round mode %d unknown", d->round_mode);
    Canon c = canonicalise(*d);
    if (c.count == 0)
        return HIPQ_OK;
    HIPQ_REQUIRE(in && scale && zp && out, "null tensor pointer");
    hipStream_t s = as_stream(stream);
    if (vec4_ok(*d, c, in, out))
    {
        uint32_t groups = static_cast<uint32_t>(c.count / 4);
        const bool few = is_short(groups);
        const unsigned step = 256 * (few ? 1 : kQuantUnroll);
        unsigned blocks = (groups + step - 1) / step;
        RunView v = make_view(c);
        bool rne = d->round_mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN;
        bool uniform = row_uniform(c);
#define LAUNCH_Q4_U(QT, RNE, UNI, U)                                                                                                                                                     \
    quantize_vec4_kernel<QT, RNE, UNI, U><<<blocks, 256, 0, s>>>(static_cast<const f32x4*>(in), static_cast<const float*>(scale), static_cast<const QT*>(zp), static_cast<uint32_t*>(out), \
                                                                 groups, v, d->round_mode)
#define LAUNCH_Q4(QT, RNE, UNI) (few ? LAUNCH_Q4_U(QT, RNE, UNI, 1) : LAUNCH_Q4_U(QT, RNE, UNI, kQuantUnroll))
#define LAUNCH_Q4_T(QT)                                                                            \
    do                                                                                             \
    {                                                                                              \
        if (rne && uniform)                                                                        \
            LAUNCH_Q4(QT, true, true);                                                             \
        else if (rne)                                                                              \
            LAUNCH_Q4(QT, true, false);                                                            \
        else if (uniform)                                                                          \
            LAUNCH_Q4(QT, false, true);                                                            \
        else                                                                                       \
            LAUNCH_Q4(QT, false, false);                                                           \
    } while (0)
        if (d->quant_t == HIPQ_I8)
            LAUNCH_Q4_T(int8_t);
        else
            LAUNCH_Q4_T(uint8_t);
#undef LAUNCH_Q4_T
#undef LAUNCH_Q4
#undef LAUNCH_Q4_U
        return check_launch("quantize_vec4");
    }
    if (ragged_ok(*d, c, in, out))
    {
        const RaggedView v = make_ragged_view(c);
        const bool rne = d->round_mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN;
#define LAUNCH_QR(QT, RNE, FORM, U)                                                                                                                                           \
    quantize_ragged_kernel<QT, RNE, FORM, U><<<ragged_blocks(v, U), 256, 0, s>>>(static_cast<const float*>(in), static_cast<const float*>(scale), static_cast<const QT*>(zp), \
                                                                                 static_cast<QT*>(out), v, d->round_mode)
#define LAUNCH_QR_U(QT, RNE, FORM) (is_short(v.groups) ? LAUNCH_QR(QT, RNE, FORM, 1) : LAUNCH_QR(QT, RNE, FORM, kQuantUnroll))
#define LAUNCH_QR_F(QT, FORM) (rne ? LAUNCH_QR_U(QT, true, FORM) : LAUNCH_QR_U(QT, false, FORM))
#define LAUNCH_QR_T(FORM) (d->quant_t == HIPQ_I8 ? LAUNCH_QR_F(int8_t, FORM) : LAUNCH_QR_F(uint8_t, FORM))
        switch (ragged_form(v))
        {
        case RAGGED_STEP: LAUNCH_QR_T(RAGGED_STEP); break;
        case RAGGED_LANE: LAUNCH_QR_T(RAGGED_LANE); break;
        case RAGGED_EACH: LAUNCH_QR_T(RAGGED_EACH); break;
        }
#undef LAUNCH_QR_T
#undef LAUNCH_QR_F
#undef LAUNCH_QR_U
#undef LAUNCH_QR
        return check_launch("quantize_ragged");
    }
    DimInfo di = dim_info(*d);
    unsigned blocks = generic_blocks(c.count);
#define LAUNCH_QG(RT, QT)                                                                          \
    quantize_generic_kernel<RT, QT><<<blocks, 256, 0, s>>>(static_cast<const RT*>(in),             \
                                                           static_cast<const RT*>(scale),          \
                                                           static_cast<const QT*>(zp),             \
                                                           static_cast<QT*>(out),                  \
                                                           c.count,                                \
                                                           di,                                     \
                                                           d->round_mode)
    if (d->real_t == HIPQ_F32)
    {
        if (d->quant_t == HIPQ_U8)
            LAUNCH_QG(float, uint8_t);
        else if (d->quant_t == HIPQ_I8)
            LAUNCH_QG(float, int8_t);
        else
            LAUNCH_QG(float, int32_t);
    }
    else
    {
        if (d->quant_t == HIPQ_U8)
            LAUNCH_QG(double, uint8_t);
        else if (d->quant_t == HIPQ_I8)
            LAUNCH_QG(double, int8_t);
        else
            LAUNCH_QG(double, int32_t);
    }
#undef LAUNCH_QG
    return check_launch("quantize_generic");
}

int hipq_dequantize(const hipq_quant_desc_t* d, const void* in, const void* scale, const void* zp, void* out, void* stream)
{
    int rc = check_desc(d);
    if (rc)
        return rc;
    Canon c = canonicalise(*d);
    if (c.count == 0)
        return HIPQ_OK;
    HIPQ_REQUIRE(in && scale && zp && out, "null tensor pointer");
    hipStream_t s = as_stream(stream);
    if (vec4_ok(*d, c, out, in))
    {
        uint32_t groups = static_cast<uint32_t>(c.count / 4);
        const bool few = is_short(groups);
        const unsigned step = 256 * (few ? 1 : kDequantUnroll);
        unsigned blocks = (groups + step - 1) / step;
        RunView v = make_view(c);
        bool uniform = row_uniform(c);
#define LAUNCH_D4_U(QT, UNI, U)                                                                                                                                                            \
    dequantize_vec4_kernel<QT, UNI, U><<<blocks, 256, 0, s>>>(static_cast<const uint32_t*>(in), static_cast<const float*>(scale), static_cast<const QT*>(zp), static_cast<f32x4*>(out), groups, v)
#define LAUNCH_D4(QT, UNI) (few ? LAUNCH_D4_U(QT, UNI, 1) : LAUNCH_D4_U(QT, UNI, kDequantUnroll))
        if (d->quant_t == HIPQ_I8)
        {
            if (uniform)
                LAUNCH_D4(int8_t, true);
            else
                LAUNCH_D4(int8_t, false);
        }
        else
        {
            if (uniform)
                LAUNCH_D4(uint8_t, true);
            else
                LAUNCH_D4(uint8_t, false);
        }
#undef LAUNCH_D4
#undef LAUNCH_D4_U
        return check_launch("dequantize_vec4");
    }
    if (ragged_ok(*d, c, out, in))
    {
        const RaggedView v = make_ragged_view(c);
#define LAUNCH_DR(QT, FORM, U)                                                                                                                                              \
    dequantize_ragged_kernel<QT, FORM, U><<<ragged_blocks(v, U), 256, 0, s>>>(static_cast<const QT*>(in), static_cast<const float*>(scale), static_cast<const QT*>(zp), \
                                                                              static_cast<float*>(out), v)
#define LAUNCH_DR_U(QT, FORM) (is_short(v.groups) ? LAUNCH_DR(QT, FORM, 1) : LAUNCH_DR(QT, FORM, kDequantUnroll))
#define LAUNCH_DR_T(FORM) (d->quant_t == HIPQ_I8 ? LAUNCH_DR_U(int8_t, FORM) : LAUNCH_DR_U(uint8_t, FORM))
        switch (ragged_form(v))
        {
        case RAGGED_STEP: LAUNCH_DR_T(RAGGED_STEP); break;
        case RAGGED_LANE: LAUNCH_DR_T(RAGGED_LANE); break;
        case RAGGED_EACH: LAUNCH_DR_T(RAGGED_EACH); break;
        }
#undef LAUNCH_DR_T
#undef LAUNCH_DR_U
#undef LAUNCH_DR
        return check_launch("dequantize_ragged");
    }
    DimInfo di = dim_info(*d);
    unsigned blocks = generic_blocks(c.count);
#define LAUNCH_DG(QT, RT)                                                                          \
    dequantize_generic_kernel<QT, RT><<<blocks, 256, 0, s>>>(static_cast<const QT*>(in),           \
                                                             static_cast<const RT*>(scale),        \
                                                             static_cast<const QT*>(zp),           \
                                                             static_cast<RT*>(out),                \
                                                             c.count,                              \
                                                             di)
    if (d->real_t == HIPQ_F32)
    {
        if (d->quant_t == HIPQ_U8)
            LAUNCH_DG(uint8_t, float);
        else if (d->quant_t == HIPQ_I8)
            LAUNCH_DG(int8_t, float);
        else
            LAUNCH_DG(int32_t, float);
    }
    else
    {
        if (d->quant_t == HIPQ_U8)
            LAUNCH_DG(uint8_t, double);
        else if (d->quant_t == HIPQ_I8)
            LAUNCH_DG(int8_t, double);
        else
            LAUNCH_DG(int32_t, double);
    }
#undef LAUNCH_DG
    return check_launch("dequantize_generic");
}
}
