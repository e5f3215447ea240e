// Entry points of the quantized convolution / dot family: argument checks, choice between the
// MFMA kernels and the direct kernels, layout conversion through the device workspace.
#include <cstdlib>

#include <cstring>

#include "hipq_common.h"

namespace hipq
{
    static bool is_quant8(int t) { return t == HIPQ_U8 || t == HIPQ_I8; }

    static int check_conv_types(const ConvGeom& g, bool fused)
    {
        // INTERPRETER combinations: int_executable.hpp:1461-1549 (data is u8 there); i8 data is
        // accepted as well because the oneDNN-backed fused ops take it.
        if (!is_quant8(g.data_t) || !is_quant8(g.filter_t))
            return fail(HIPQ_ERR_UNSUPPORTED, "data and filter must be u8 or i8");
        if (!is_quant8(g.out_t) && g.out_t != HIPQ_I32)
            return fail(HIPQ_ERR_UNSUPPORTED, "convolution output must be i8, u8 or i32");
        if (fused && g.filter_t != HIPQ_I8)
            return fail(HIPQ_ERR_UNSUPPORTED, "fused convolutions take i8 filters");
        return HIPQ_OK;
    }

    // Runs the convolution with whatever layouts the descriptor names.
    static int run_conv(const ConvGeom& whole,
                        const void* data,
                        const void* filter,
                        const void* packed,
                        const ZeroPoints& zp,
                        Epilogue epi,
                        void* out,
                        hipStream_t s)
    {
        // the MFMA kernels have no fused-policy instantiation with int32 output (no nGraph op asks for one)
        RowPack rp;
        // a first layer the band kernel takes whole: it reads the [N][C][H][W] bytes itself
        if (packed && (reinterpret_cast<uintptr_t>(data) & 3) == 0 && conv_rowpack_eligible(whole, &rp) && conv_stem_eligible(whole, epi, zp, nullptr))
            return launch_conv_stem(whole, data, packed, zp, epi, nullptr, out, s);
        if (packed && conv_rowpack_eligible(whole, &rp))
        {
            // a first layer's three or four channels: a copy with the padding materialised, whose
            // filter rows are single 32-byte runs, then the tile kernel that loads straight into LDS
            void* ws = nullptr;
            int rc = workspace(align_up(static_cast<size_t>(whole.N * rp.Hp * rp.Wp * 4), 256), s, &ws);
            if (rc)
                return rc;
            rc = launch_stage_rows(whole, rp, data, ws, zp.data_zp, zp.data_t, s);
            if (rc)
                return rc;
            return launch_conv_rowpack(whole, rp, ws, packed, zp, epi, out, s);
        }
        ConvGeom padded;
        // (widths above 16 that are no multiple of it: tensors that start on no 16-byte boundary keep the direct
        // kernel, as products do, and so does the entry point that allocates nothing where the copy would not
        // fit its array)
        const bool aligned = ((reinterpret_cast<uintptr_t>(packed) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(epi.sum_in)) & 15) == 0;
        const bool pad =
            packed && !conv_mfma_eligible(whole) && conv_pad_eligible(whole, &padded) && (whole.C < 16 || (aligned && workspace_holds(static_cast<size_t>(padded.in_count()) + 256)));
        if (!packed || (!pad && !conv_mfma_eligible(whole)) || (epi.mode == EPI_FUSED && whole.out_t == HIPQ_I32))
            return launch_conv_direct(whole, data, filter, zp, epi, out, s);
        // the geometry the MFMA kernels see: channels in whole 16-byte pieces
        const ConvGeom& g = pad ? padded : whole;

        const int64_t in_sp = g.in[1] * g.in[2];
        const bool out_ncx = g.out_layout == HIPQ_LAYOUT_NCX && g.K > 1;
        const bool tr_in = !pad && g.data_layout == HIPQ_LAYOUT_NCX && g.C > 1;
        const size_t tr_bytes = pad || tr_in ? align_up(static_cast<size_t>(g.in_count()), 256) : 0;
        // channels-last pixels of any width, where reading them as they lie costs less than the copy
        if (pad && conv_ragged_preferred(whole, g, epi, out_ncx) && !conv_pw64_eligible(g, epi, zp) && !conv_regw_eligible(g, out_ncx))
            return launch_conv_ragged(whole, g, data, packed, zp, epi, out, out_ncx, s);
        const void* x = data;
        uint8_t* ws = nullptr;
        auto scratch = [&]() {
            void* p = nullptr;
            const int rc = tr_bytes ? workspace(tr_bytes, s, &p) : HIPQ_OK;
            ws = static_cast<uint8_t*>(p);
            return rc;
        };
        if (pad)
        {
            // the channels-last copy with the missing channels of every pixel at the data zero point (they
            // meet zero weights; as the zero point they also vanish on the exact path for a non-zero
            // filter zero point)
            int rc = scratch();
            if (rc)
                return rc;
            if (whole.C < 16)
                rc = launch_pad_channels(data, ws, g.N, in_sp, whole.C, whole.data_layout == HIPQ_LAYOUT_NCX, zp.data_zp, zp.data_t, s);
            else if (whole.data_layout == HIPQ_LAYOUT_NCX)
                rc = launch_transpose_pad(data, ws, g.N, whole.C, in_sp, g.C, zp.data_zp, zp.data_t, s);
            else
                rc = launch_pad_rows(data, ws, g.N * in_sp, whole.C, g.C, zp.data_zp, zp.data_t, s);
            if (rc)
                return rc;
            x = ws;
        }

        // layers bound by HBM traffic that widen 64 channels: weights in registers, loads a tile ahead
        if (conv_pw64_eligible(g, epi, zp))
            return launch_conv_pw64(g, x, packed, epi, out, s);
        if (conv_stream_eligible(g, epi, zp))
            return launch_conv_stream(g, x, packed, epi, out, s);

        // 3x3 layers over 64 channels with an NCHW output keep their filter in registers and read the
        // input in whichever layout it has: no transposition, no scratch
        if (conv_regw_eligible(g, out_ncx))
            return launch_conv_regw(g, x, packed, zp, epi, out, true, s);

        // The other kernels read channels-last data; an NCHW input is transposed through the workspace.
        // The output is written directly in either layout (sum_in is indexed like the output).
        if (!pad)
        {
            const int rc = scratch();
            if (rc)
                return rc;
        }
        if (tr_in)
        {
            HIPQ_REQUIRE(g.N <= 65535, "batch %lld beyond 65535", (long long)g.N);
            const int rc = in_sp % 16 == 0 ? launch_transpose(data, ws, g.N, g.C, in_sp, 1, s) : launch_transpose_pad(data, ws, g.N, g.C, in_sp, g.C, nullptr, HIPQ_U8, s);
            if (rc)
                return rc;
            x = ws;
        }
        // layers whose filter fits in LDS take the band kernel (HIPQ_NO_BAND=1 forces the generic one)
        const bool no_band = getenv("HIPQ_NO_BAND") != nullptr;
        // (a 1 x 1 filter over every pixel, 8-bit channels-last output in whole 16-byte rows: the data
        // is a row matrix and the tile kernels that load it straight into LDS are faster -- 64 -> 64
        // channels at 56 x 56, batch 128: 15.8 us against 23 us)
        const bool row_matrix = !out_ncx && g.taps() == 1 && g.st[1] == 1 && g.st[2] == 1 && g.pb[1] == 0 && g.pb[2] == 0 && g.out[1] == g.in[1] && g.out[2] == g.in[2] &&
                                (g.out_t == HIPQ_U8 || g.out_t == HIPQ_I8) && g.K % 16 == 0 && getenv("HIPQ_NO_DMA") == nullptr && getenv("HIPQ_NO_PIPE") == nullptr;
        // (nor layers too small to fill the chip)
        if (!no_band && !row_matrix && conv_band_eligible(g, out_ncx) && !conv_wk_preferred(g, epi.out_t, out_ncx))
            return launch_conv_band(g, x, packed, zp, epi, out, out_ncx, s);
        return launch_conv_mfma(g, x, packed, zp, epi, out, out_ncx, s);
    }

    static int fused_epilogue(const hipq_fused_desc_t* f,
                              int out_t,
                              int64_t channels,
                              const int32_t* bias,
                              const void* sum_in,
                              const float* scale,
                              const float* sum_scale,
                              Epilogue* e)
    {
        HIPQ_REQUIRE(f, "fused descriptor is null");
        HIPQ_REQUIRE(scale, "scale is null");
        HIPQ_REQUIRE(f->scale_count == 1 || f->scale_count == channels,
                     "scale_count %lld is neither 1 nor the channel count %lld",
                     (long long)f->scale_count,
                     (long long)channels);
        HIPQ_REQUIRE(!f->has_bias || bias, "has_bias set but bias is null");
        HIPQ_REQUIRE(!f->has_sum || (sum_in && sum_scale), "has_sum set but sum_in / sum_scale is null");
        if (f->has_sum && !is_quant8(f->sum_t))
            return fail(HIPQ_ERR_UNSUPPORTED, "sum input must be u8 or i8");
        memset(e, 0, sizeof(*e));
        e->mode = EPI_FUSED;
        e->out_t = out_t;
        e->bias = f->has_bias ? bias : nullptr;
        e->scale = scale;
        e->per_channel = f->scale_count > 1;
        e->sum_in = f->has_sum ? sum_in : nullptr;
        e->sum_scale = f->has_sum ? sum_scale : nullptr;
        e->sum_t = f->sum_t;
        e->relu = f->with_relu;
        return HIPQ_OK;
    }

    static int dot_pack(const hipq_dot_desc_t& d, const void* b, void* packed, bool with_fragments, hipStream_t s);

    // The product the MFMA kernels see: reductions in whole 16-byte pieces of a row.  A reduction that is
    // not is padded to whole 64-byte steps -- zero weights in the packed operand, a padded copy of the
    // rows of `a` in the workspace.  Below 64 there is less to multiply than to pad: the direct kernel.
    static bool dot_is_padded(const hipq_dot_desc_t& d) { return d.K >= 64 && d.K % 16 != 0; }
    static hipq_dot_desc_t dot_seen(const hipq_dot_desc_t& d)
    {
        hipq_dot_desc_t p = d;
        if (dot_is_padded(d))
            p.K = static_cast<int64_t>(align_up(static_cast<size_t>(d.K), 64));
        return p;
    }

    // Layout of a packed dot operand: [N][K] weights (only when the caller's are [K][N] or need padding),
    // the column sums, and -- for products the weight-streaming kernels take -- the weights once more in
    // MFMA fragment order.  Each part starts on a 256-byte boundary.
    static bool dot_blob_has_weights(const hipq_dot_desc_t& d) { return d.b_layout == HIPQ_B_KN || dot_is_padded(d); }
    static size_t dot_blob_weights(const hipq_dot_desc_t& d) { return dot_blob_has_weights(d) ? align_up(static_cast<size_t>(d.N * dot_seen(d).K), 256) : 0; }
    static size_t dot_blob_sums(const hipq_dot_desc_t& d) { return align_up(static_cast<size_t>(d.N) * sizeof(int32_t), 256); }

    // Operands of the MFMA dot: the rows of `a` (padded through the workspace where the reduction is) and
    // the weights [N,K] with their column sums, either prepacked or built in the workspace
    // (built on the fly there is no fragment-ordered copy: making one costs more than it saves a call)
    struct DotOperands
    {
        hipq_dot_desc_t d; // as the kernels see it
        const void* a;
        const void* w;
        const void* wfrag;
        const int32_t* wsum;
        int64_t a_row; // bytes of a row of `a` where it stays unpadded, 0: the padded reduction
    };
    static size_t dot_padded_rows_bytes(const hipq_dot_desc_t& d) { return dot_is_padded(d) ? align_up(static_cast<size_t>(d.M * dot_seen(d).K), 256) : 0; }

    // scratch (may be null: the workspace): where the copies go, for a caller that holds a part of the
    // workspace itself
    static int dot_operands(const hipq_dot_desc_t& d, const void* a, const void* b, const void* packed, const ZeroPoints& zp, const Epilogue& epi, DotOperands* o, hipStream_t s,
                            uint8_t* scratch = nullptr)
    {
        o->d = dot_seen(d);
        o->a = a;
        o->wfrag = nullptr;
        const size_t wbytes = dot_blob_weights(d);
        const size_t blob_bytes = packed ? 0 : wbytes + dot_blob_sums(d);
        const bool in_place = dot_is_padded(d) && dot_ragged_preferred(o->d, d.K, epi);
        o->a_row = in_place ? d.K : 0;
        const size_t a_bytes = in_place ? 0 : dot_padded_rows_bytes(d);
        const uint8_t* blob = static_cast<const uint8_t*>(packed);
        if (blob_bytes + a_bytes)
        {
            uint8_t* ws = scratch;
            int rc = ws ? HIPQ_OK : workspace(blob_bytes + a_bytes, s, reinterpret_cast<void**>(&ws));
            if (rc)
                return rc;
            if (a_bytes)
            {
                // (the bytes behind a row's end meet zero weights; as the zero point they also vanish on the
                // exact path for a non-zero weight zero point)
                rc = launch_pad_rows(a, ws + blob_bytes, d.M, d.K, o->d.K, zp.data_zp, zp.data_t, s);
                if (rc)
                    return rc;
                o->a = ws + blob_bytes;
            }
            if (blob_bytes)
            {
                rc = dot_pack(d, b, ws, false, s);
                if (rc)
                    return rc;
                blob = ws;
            }
        }
        if (packed && dot_fragments_eligible(o->d))
            o->wfrag = blob + wbytes + dot_blob_sums(d);
        o->w = dot_blob_has_weights(d) ? static_cast<const void*>(blob) : b;
        o->wsum = reinterpret_cast<const int32_t*>(blob + wbytes);
        return HIPQ_OK;
    }

    static int run_dot(const hipq_dot_desc_t& d,
                       const void* a,
                       const void* b,
                       const void* packed,
                       const ZeroPoints& zp,
                       const Epilogue& epi,
                       void* out,
                       hipStream_t s,
                       uint8_t* scratch = nullptr)
    {
        if (d.M == 0 || d.N == 0)
            return HIPQ_OK;
        HIPQ_REQUIRE(out && (d.K == 0 || (a && b)), "null tensor pointer");
        // (operands that the padded copies replace may start anywhere, the packed weights they are read from may not)
        const bool copied = dot_is_padded(d);
        const uintptr_t misaligned = reinterpret_cast<uintptr_t>(out) | (copied ? reinterpret_cast<uintptr_t>(packed) : reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b));
        // Padding and packing a reduction on the fly is three launches ahead of the product: from 2^24
        // multiply-adds on, where the direct kernel takes ten times as long as those
        if (!dot_mfma_eligible(dot_seen(d)) || (misaligned & 15) || (copied && !packed && d.M * d.N < (1ll << 31) && d.M * d.N * d.K < (1ll << 24)))
            return launch_dot_direct(d, a, b, zp, epi, out, s);
        DotOperands o;
        const int rc = dot_operands(d, a, b, packed, zp, epi, &o, s, scratch);
        if (rc)
            return rc;
        return launch_dot_mfma(o.d, o.a, o.w, o.wsum, zp, epi, out, s, o.wfrag, o.a_row);
    }

    static int dot_pack(const hipq_dot_desc_t& d, const void* b, void* packed, bool with_fragments, hipStream_t s)
    {
        uint8_t* blob = static_cast<uint8_t*>(packed);
        const void* w = b;
        const size_t wbytes = dot_blob_weights(d);
        const hipq_dot_desc_t seen = dot_seen(d);
        if (dot_blob_has_weights(d))
        {
            // [K][N] -> [N][K], or [N][K] rows padded
            const int rc = d.b_layout != HIPQ_B_KN ? launch_pad_rows(b, blob, d.N, d.K, seen.K, nullptr, HIPQ_I8, s)
                           : d.N % 16 == 0 && seen.K == d.K ? launch_transpose(b, blob, 1, d.K, d.N, 1, s)
                                                            : launch_transpose_pad(b, blob, 1, d.K, d.N, seen.K, nullptr, HIPQ_I8, s);
            if (rc)
                return rc;
            w = blob;
        }
        const int rc = launch_row_sums_i8(w, d.N, seen.K, reinterpret_cast<int32_t*>(blob + wbytes), s);
        if (rc || !with_fragments || !dot_fragments_eligible(seen))
            return rc;
        return launch_pack_dot_fragments(w, d.N, seen.K, blob + wbytes + dot_blob_sums(d), s);
    }
}

using namespace hipq;

extern "C" {

int hipq_conv_infer_output(hipq_conv_desc_t* d)
{
    HIPQ_REQUIRE(d, "descriptor is null");
    HIPQ_REQUIRE(d->n_spatial >= 1 && d->n_spatial <= HIPQ_MAX_SPATIAL, "n_spatial %d out of range", d->n_spatial);
    for (int i = 0; i < d->n_spatial; ++i)
    {
        HIPQ_REQUIRE(d->in_sp[i] >= 1 && d->f_sp[i] >= 1 && d->stride[i] >= 1 && d->dilation[i] >= 1 && d->data_dilation[i] >= 1,
                     "non-positive extent, stride or dilation on spatial axis %d", i);
        int64_t in_eff = (d->in_sp[i] - 1) * d->data_dilation[i] + 1 + d->pad_below[i] + d->pad_above[i];
        int64_t f_eff = (d->f_sp[i] - 1) * d->dilation[i] + 1;
        HIPQ_REQUIRE(in_eff >= f_eff, "window larger than padded data on spatial axis %d", i);
        d->out_sp[i] = (in_eff - f_eff) / d->stride[i] + 1;
    }
    return HIPQ_OK;
}

int hipq_quantized_convolution(const hipq_conv_desc_t* desc,
                               const void* data,
                               const void* filter,
                               const void* packed_filter,
                               const float* data_scale,
                               const void* data_zp,
                               const float* filter_scale,
                               const void* filter_zp,
                               const float* out_scale,
                               const void* out_zp,
                               void* out,
                               void* stream)
{
    ConvGeom g;
    int rc = make_geom(desc, &g);
    if (rc)
        return rc;
    rc = check_conv_types(g, false);
    if (rc)
        return rc;
    HIPQ_REQUIRE(data && filter && out, "null tensor pointer");
    HIPQ_REQUIRE(data_scale && data_zp && filter_scale && filter_zp && out_scale && out_zp, "null scale or zero point");
    Epilogue e;
    memset(&e, 0, sizeof(e));
    e.mode = EPI_INTERP;
    e.out_t = g.out_t;
    e.s_data = data_scale;
    e.s_filter = filter_scale;
    e.s_out = out_scale;
    e.out_zp = out_zp;
    ZeroPoints zp{data_zp, filter_zp, g.data_t, g.filter_t};
    return run_conv(g, data, filter, packed_filter, zp, e, out, as_stream(stream));
}

int hipq_quantized_convolution_noalloc(const hipq_conv_desc_t* desc,
                                       const void* data,
                                       const void* filter,
                                       const void* packed_filter,
                                       const float* data_scale,
                                       const void* data_zp,
                                       const float* filter_scale,
                                       const void* filter_zp,
                                       const float* out_scale,
                                       const void* out_zp,
                                       void* out,
                                       void* stream)
{
    // same kernels, same choices; whatever scratch they need comes out of the fixed per-device array
    int rc = noalloc_begin();
    if (rc)
        return rc;
    rc = hipq_quantized_convolution(desc, data, filter, packed_filter, data_scale, data_zp, filter_scale, filter_zp, out_scale, out_zp, out, stream);
    noalloc_end();
    return rc;
}

int hipq_quantized_convolution_fused(const hipq_conv_desc_t* desc,
                                     const hipq_fused_desc_t* fused,
                                     const void* data,
                                     const void* filter,
                                     const void* packed_filter,
                                     const int32_t* bias,
                                     const void* sum_in,
                                     const float* scale,
                                     const float* sum_scale,
                                     void* out,
                                     void* stream)
{
    ConvGeom g;
    int rc = make_geom(desc, &g);
    if (rc)
        return rc;
    rc = check_conv_types(g, true);
    if (rc)
        return rc;
    HIPQ_REQUIRE(data && filter && out, "null tensor pointer");
    Epilogue e;
    rc = fused_epilogue(fused, g.out_t, g.K, bias, sum_in, scale, sum_scale, &e);
    if (rc)
        return rc;
    ZeroPoints zp{nullptr, nullptr, g.data_t, g.filter_t};
    return run_conv(g, data, filter, packed_filter, zp, e, out, as_stream(stream));
}

// MaxPool over the output of a fused convolution, as the pair of descriptors the two calls would take
static int conv_pool_pair(const hipq_conv_desc_t* desc, const hipq_fused_desc_t* fused, const hipq_pool_desc_t* pool, ConvGeom* g, PoolFuse* pf)
{
    int rc = make_geom(desc, g);
    if (rc)
        return rc;
    rc = check_conv_types(*g, true);
    if (rc)
        return rc;
    HIPQ_REQUIRE(fused && pool, "descriptor is null");
    if (g->in[0] != 1 || pool->op != HIPQ_POOL_MAX || pool->n_spatial != 2 || desc->n_spatial != 2 || pool->dtype != g->out_t || pool->layout != g->out_layout || pool->N != g->N ||
        pool->C != g->K || pool->in_sp[0] != g->out[1] || pool->in_sp[1] != g->out[2] || fused->has_sum)
        return fail(HIPQ_ERR_UNSUPPORTED, "not a 2-D MaxPool over this convolution's output");
    hipq_pool_desc_t pd = *pool;
    rc = hipq_pool_infer_output(&pd);
    if (rc)
        return rc;
    pf->wh = pool->window[0];
    pf->ww = pool->window[1];
    pf->sh = pool->stride[0];
    pf->sw = pool->stride[1];
    pf->pt = pool->pad_below[0];
    pf->pl = pool->pad_below[1];
    pf->out_h = pd.out_sp[0];
    pf->out_w = pd.out_sp[1];
    return HIPQ_OK;
}

int hipq_conv_max_pool_fusable(const hipq_conv_desc_t* desc, const hipq_fused_desc_t* fused, const hipq_pool_desc_t* pool)
{
    ConvGeom g;
    PoolFuse pf;
    if (!desc || !fused || !pool || conv_pool_pair(desc, fused, pool, &g, &pf) != HIPQ_OK)
        return 0;
    Epilogue e;
    memset(&e, 0, sizeof(e));
    e.mode = EPI_FUSED;
    e.out_t = g.out_t;
    ZeroPoints zp{nullptr, nullptr, g.data_t, g.filter_t};
    RowPack rp;
    return conv_rowpack_eligible(g, &rp) && conv_stem_eligible(g, e, zp, &pf) ? 1 : 0;
}

int hipq_quantized_convolution_fused_max_pool(const hipq_conv_desc_t* desc,
                                              const hipq_fused_desc_t* fused,
                                              const hipq_pool_desc_t* pool,
                                              const void* data,
                                              const void* packed_filter,
                                              const int32_t* bias,
                                              const float* scale,
                                              void* out,
                                              void* stream)
{
    ConvGeom g;
    PoolFuse pf;
    int rc = conv_pool_pair(desc, fused, pool, &g, &pf);
    if (rc)
        return rc;
    HIPQ_REQUIRE(data && packed_filter && out, "null tensor pointer");
    Epilogue e;
    rc = fused_epilogue(fused, g.out_t, g.K, bias, nullptr, scale, nullptr, &e);
    if (rc)
        return rc;
    ZeroPoints zp{nullptr, nullptr, g.data_t, g.filter_t};
    RowPack rp;
    if (!conv_rowpack_eligible(g, &rp) || !conv_stem_eligible(g, e, zp, &pf))
        return fail(HIPQ_ERR_UNSUPPORTED, "this convolution / MaxPool pair has no fused kernel (hipq_conv_max_pool_fusable is 0)");
    return launch_conv_stem(g, data, packed_filter, zp, e, &pf, out, as_stream(stream));
}

// the layers of a chain of pointwise convolutions, pointers and all; `sum` stands for the residual or the shortcut's data
static int chain_layers(const hipq_pointwise_layer_t* widen, const hipq_pointwise_layer_t* shortcut, const hipq_pointwise_layer_t* narrow, const void* sum, const float* sum_scale, ConvGeom (&g)[3],
                        Epilogue (&e)[3])
{
    const hipq_pointwise_layer_t* const layers[3] = {widen, shortcut, narrow};
    HIPQ_REQUIRE(widen && narrow, "layer is null");
    for (int i = 0; i < 3; ++i)
    {
        if (!layers[i])
            continue;
        int rc = make_geom(layers[i]->conv, &g[i]);
        if (rc)
            return rc;
        rc = check_conv_types(g[i], true);
        if (rc)
            return rc;
        if (i != 0 && layers[i]->fused && layers[i]->fused->has_sum)
            return fail(HIPQ_ERR_UNSUPPORTED, "the narrowing layer and the shortcut of a pointwise chain have no residual");
        rc = fused_epilogue(layers[i]->fused, g[i].out_t, g[i].K, layers[i]->bias, i == 0 ? sum : nullptr, layers[i]->scale, i == 0 ? sum_scale : nullptr, &e[i]);
        if (rc)
            return rc;
    }
    if (!widen->fused->has_sum || !conv_chain_eligible(g[0], e[0], shortcut ? &g[1] : nullptr, shortcut ? &e[1] : nullptr, g[2], e[2]))
        return fail(HIPQ_ERR_UNSUPPORTED, "these pointwise layers have no common kernel (hipq_pointwise_chain_fusable is 0)");
    return HIPQ_OK;
}

int hipq_pointwise_chain_fusable(const hipq_pointwise_layer_t* widen, const hipq_pointwise_layer_t* shortcut, const hipq_pointwise_layer_t* narrow)
{
    if (!widen || !narrow)
        return 0;
    // (only what the descriptors say counts: any address stands for a tensor that will be there)
    static const int32_t there[4] = {};
    auto with = [](const hipq_pointwise_layer_t* l) {
        hipq_pointwise_layer_t r = *l;
        r.bias = there;
        r.scale = reinterpret_cast<const float*>(there);
        return r;
    };
    const hipq_pointwise_layer_t w = with(widen), s = shortcut ? with(shortcut) : w, n = with(narrow);
    ConvGeom g[3];
    Epilogue e[3];
    return chain_layers(&w, shortcut ? &s : nullptr, &n, there, reinterpret_cast<const float*>(there), g, e) == HIPQ_OK ? 1 : 0;
}

int hipq_pointwise_chain(const hipq_pointwise_layer_t* widen,
                         const hipq_pointwise_layer_t* shortcut,
                         const hipq_pointwise_layer_t* narrow,
                         const void* sum_in,
                         const float* sum_scale,
                         void* wide_out,
                         void* narrow_out,
                         void* stream)
{
    HIPQ_REQUIRE(!shortcut || !sum_in, "either a residual or a shortcut");
    ConvGeom g[3];
    Epilogue e[3];
    const int rc = chain_layers(widen, shortcut, narrow, shortcut ? shortcut->data : sum_in, sum_scale, g, e);
    if (rc)
        return rc;
    HIPQ_REQUIRE(widen->data && widen->packed_filter && narrow->packed_filter && (!shortcut || shortcut->packed_filter) && wide_out && narrow_out, "null tensor pointer");
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (!aligned(widen->data) || !aligned(widen->packed_filter) || !aligned(e[0].sum_in) || !aligned(narrow->packed_filter) || (shortcut && !aligned(shortcut->packed_filter)) || !aligned(wide_out) ||
        !aligned(narrow_out))
        return fail(HIPQ_ERR_UNSUPPORTED, "tensors of a pointwise chain must be 16-byte aligned");
    // A workgroup writes its pixels of both results while others have not read theirs: an output may stand on an input only pixel by pixel
    const int64_t pixels = g[0].N * g[0].in[1] * g[0].in[2];
    auto clash = [&](const void* out, int64_t out_row, const void* in, int64_t in_row) {
        const uintptr_t o = reinterpret_cast<uintptr_t>(out), i = reinterpret_cast<uintptr_t>(in);
        return o < i + pixels * in_row && i < o + pixels * out_row && !(o == i && out_row == in_row);
    };
    const int64_t sum_row = shortcut ? g[1].C : g[0].K;
    if (clash(wide_out, g[0].K, widen->data, g[0].C) || clash(wide_out, g[0].K, e[0].sum_in, sum_row) || clash(narrow_out, g[2].K, widen->data, g[0].C) ||
        clash(narrow_out, g[2].K, e[0].sum_in, sum_row) || clash(narrow_out, g[2].K, wide_out, g[0].K))
        return fail(HIPQ_ERR_UNSUPPORTED, "results of a pointwise chain overlap its inputs or each other");
    return launch_conv_chain(g[0], e[0], widen->data, widen->packed_filter, shortcut ? &g[1] : nullptr, shortcut ? &e[1] : nullptr, shortcut ? shortcut->packed_filter : nullptr, g[2], e[2],
                             narrow->packed_filter, wide_out, narrow_out, as_stream(stream));
}

size_t hipq_dot_packed_bytes(const hipq_dot_desc_t* d)
{
    if (!d || !dot_mfma_eligible(dot_seen(*d)))
        return 0;
    const hipq_dot_desc_t seen = dot_seen(*d);
    return dot_blob_weights(*d) + dot_blob_sums(*d) + (dot_fragments_eligible(seen) ? dot_fragment_bytes(seen) : 0);
}

int hipq_dot_pack(const hipq_dot_desc_t* d, const void* b, void* packed, void* stream)
{
    HIPQ_REQUIRE(d && b && packed, "null pointer");
    if (!dot_mfma_eligible(dot_seen(*d)))
        return fail(HIPQ_ERR_UNSUPPORTED, "shape is not eligible for the MFMA path (hipq_dot_packed_bytes is 0)");
    return dot_pack(*d, b, packed, true, as_stream(stream));
}

int hipq_quantized_dot(const hipq_dot_desc_t* d,
                       const void* a,
                       const void* b,
                       const void* packed_b,
                       const float* a_scale,
                       const void* a_zp,
                       const float* b_scale,
                       const void* b_zp,
                       const float* out_scale,
                       const void* out_zp,
                       void* out,
                       void* stream)
{
    HIPQ_REQUIRE(d, "descriptor is null");
    HIPQ_REQUIRE(d->M >= 0 && d->N >= 0 && d->K >= 0, "negative extent");
    HIPQ_REQUIRE(d->b_layout == HIPQ_B_KN || d->b_layout == HIPQ_B_NK, "bad b_layout");
    if (!is_quant8(d->a_t) || !is_quant8(d->b_t) || (!is_quant8(d->out_t) && d->out_t != HIPQ_I32))
        return fail(HIPQ_ERR_UNSUPPORTED, "QuantizedDot takes u8/i8 operands and gives i8, u8 or i32");
    HIPQ_REQUIRE(a_scale && a_zp && b_scale && b_zp && out_scale && out_zp, "null scale or zero point");
    Epilogue e;
    memset(&e, 0, sizeof(e));
    e.mode = EPI_INTERP;
    e.out_t = d->out_t;
    e.s_data = a_scale;
    e.s_filter = b_scale;
    e.s_out = out_scale;
    e.out_zp = out_zp;
    ZeroPoints zp{a_zp, b_zp, d->a_t, d->b_t};
    return run_dot(*d, a, b, packed_b, zp, e, out, as_stream(stream));
}

int hipq_quantized_dot_bias(const hipq_dot_desc_t* d,
                            const hipq_fused_desc_t* fused,
                            const void* a,
                            const void* w,
                            const void* packed_w,
                            const int32_t* bias,
                            const float* scale,
                            void* out,
                            void* stream)
{
    HIPQ_REQUIRE(d, "descriptor is null");
    HIPQ_REQUIRE(d->M >= 0 && d->N >= 0 && d->K >= 0, "negative extent");
    HIPQ_REQUIRE(d->b_layout == HIPQ_B_KN || d->b_layout == HIPQ_B_NK, "bad b_layout");
    if (!is_quant8(d->a_t) || d->b_t != HIPQ_I8 || (!is_quant8(d->out_t) && d->out_t != HIPQ_F32))
        return fail(HIPQ_ERR_UNSUPPORTED, "QuantizedDotBias takes u8/i8 data, i8 weights and gives i8, u8 or f32");
    HIPQ_REQUIRE(fused && !fused->has_sum, "QuantizedDotBias has no sum input");
    Epilogue e;
    int rc = fused_epilogue(fused, d->out_t, d->N, bias, nullptr, scale, nullptr, &e);
    if (rc)
        return rc;
    ZeroPoints zp{nullptr, nullptr, d->a_t, d->b_t};
    return run_dot(*d, a, w, packed_w, zp, e, out, as_stream(stream));
}

int hipq_quantized_dot_bias_gelu_quantize(const hipq_dot_desc_t* d,
                                          const hipq_fused_desc_t* fused,
                                          const void* a,
                                          const void* w,
                                          const void* packed_w,
                                          const int32_t* bias,
                                          const float* scale,
                                          const hipq_quant_out_t* quant,
                                          void* stream)
{
    HIPQ_REQUIRE(d, "descriptor is null");
    HIPQ_REQUIRE(d->M >= 0 && d->N >= 0 && d->K >= 0, "negative extent");
    HIPQ_REQUIRE(d->b_layout == HIPQ_B_KN || d->b_layout == HIPQ_B_NK, "bad b_layout");
    if (!is_quant8(d->a_t) || d->b_t != HIPQ_I8 || d->out_t != HIPQ_F32)
        return fail(HIPQ_ERR_UNSUPPORTED, "QuantizedDotBias + Gelu + Quantize takes u8/i8 data, i8 weights and the f32 form of the product (out_t F32)");
    HIPQ_REQUIRE(fused && !fused->has_sum, "QuantizedDotBias has no sum input");
    HIPQ_REQUIRE(quant && quant->out && quant->scale, "quantized output: null pointer");
    HIPQ_REQUIRE(quant->quant_t == HIPQ_I8 || quant->quant_t == HIPQ_U8, "quantized output: i8 or u8");
    HIPQ_REQUIRE(quant->round_mode >= HIPQ_ROUND_NEAREST_TOWARD_INFINITY && quant->round_mode <= HIPQ_ROUND_DOWN, "quantized output: unknown round mode");
    if (d->M == 0 || d->N == 0)
        return HIPQ_OK;
    HIPQ_REQUIRE(d->K == 0 || (a && w), "null tensor pointer");
    {
        // workgroups write their output bytes while others still read rows of `a`
        const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), a1 = a0 + static_cast<size_t>(d->M * d->K);
        const uintptr_t o0 = reinterpret_cast<uintptr_t>(quant->out), o1 = o0 + static_cast<size_t>(d->M * d->N);
        HIPQ_REQUIRE(a1 <= o0 || o1 <= a0, "the quantized output must not overlap the input rows");
    }
    Epilogue e;
    int rc = fused_epilogue(fused, HIPQ_F32, d->N, bias, nullptr, scale, nullptr, &e);
    if (rc)
        return rc;
    hipStream_t s = as_stream(stream);
    // in the epilogue of the product, where the kernels that take it apply: the ones for products too
    // small to fill the chip, and from 257 rows on the tile kernels
    const bool q16 = (reinterpret_cast<uintptr_t>(quant->out) & 15) == 0;
    if (dot_mfma_eligible(*d) && d->K % 16 == 0 && (d->M > 256 || (packed_w && dot_gelu_wk_preferred(*d))) && (reinterpret_cast<uintptr_t>(a) & 15) == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0 && q16)
    {
        DotOperands o;
        ZeroPoints zp{nullptr, nullptr, d->a_t, d->b_t};
        rc = dot_operands(*d, a, w, packed_w, zp, e, &o, s);
        if (rc)
            return rc;
        Epilogue post = e;
        post.post_scale = quant->scale;
        post.post_zp = quant->zero_point;
        post.post_t = quant->quant_t;
        post.post_mode = quant->round_mode;
        rc = launch_rows_gelu_q8(a, d->a_t == HIPQ_U8, static_cast<const int8_t*>(o.w), o.wfrag, o.wsum, d->M, static_cast<int32_t>(d->N), static_cast<int32_t>(d->K), zp, post, quant->out, s);
        if (rc != HIPQ_ERR_UNSUPPORTED)
            return rc;
    }
    // otherwise the product into the workspace, then Gelu + Quantize from there (prepacked weights only:
    // weights packed on the fly live in the same workspace)
    if (!packed_w)
        return fail(HIPQ_ERR_UNSUPPORTED, "QuantizedDotBias + Gelu + Quantize outside the fused kernels needs prepacked weights (hipq_dot_pack)");
    float* product = nullptr;
    const size_t product_bytes = align_up(static_cast<size_t>(d->M) * static_cast<size_t>(d->N) * sizeof(float), 256);
    rc = workspace(product_bytes + dot_padded_rows_bytes(*d), s, reinterpret_cast<void**>(&product));
    if (rc)
        return rc;
    ZeroPoints zp{nullptr, nullptr, d->a_t, d->b_t};
    rc = run_dot(*d, a, w, packed_w, zp, e, product, s, reinterpret_cast<uint8_t*>(product) + product_bytes);
    if (rc)
        return rc;
    return hipq_gelu_quantize_f32(product, nullptr, quant, d->M * d->N, stream);
}
}
