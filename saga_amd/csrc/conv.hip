// Convolution entry points: argument checking, geometry, and the choice between the MFMA
// implicit-GEMM kernels and the direct fallback.
#include "stream_f32.hpp"

#include <stdlib.h>

namespace {

// 0 when the padded input is smaller than the dilated filter (C's division would truncate a negative
// numerator toward zero and report one output position)
static int conv_dim(int in, int k, int pad, int stride, int dil)
{
    const int span = in + 2 * pad - ((k - 1) * dil + 1);
    return span < 0 ? 0 : 1 + span / stride;
}

// x: (N,C,H,W)  w: (K,C/group,R,S)  y: (N,K,P,Q)
static int geometry(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                    ConvGeom *g)
{
    if(!valid_view(x) || !valid_view(w) || !valid_view(y) || !p)
        return SAGA_HIP_EINVAL;
    if(p->stride < 1 || p->pad < 0 || p->dilation < 1 || p->group < 1)
        return SAGA_HIP_EINVAL;
    g->N = x->dims[0]; g->C = x->dims[1]; g->H = x->dims[2]; g->W = x->dims[3];
    g->K = w->dims[0]; g->R = w->dims[2]; g->S = w->dims[3];
    g->pad = p->pad; g->stride = p->stride; g->dil = p->dilation; g->group = p->group;
    g->P = conv_dim(g->H, g->R, g->pad, g->stride, g->dil);
    g->Q = conv_dim(g->W, g->S, g->pad, g->stride, g->dil);
    if(g->C % g->group || g->K % g->group || w->dims[1] != g->C / g->group)
        return SAGA_HIP_ESHAPE;
    if(y->dims[0] != g->N || y->dims[1] != g->K || y->dims[2] != g->P || y->dims[3] != g->Q || g->P < 1 || g->Q < 1)
        return SAGA_HIP_ESHAPE;
    if(x->dtype != w->dtype || x->dtype != y->dtype || (x->dtype != SAGA_HALF && x->dtype != SAGA_FLOAT))
        return SAGA_HIP_EUNSUPPORTED;
    return 0;
}

static bool force_direct()
{
    static int v = -1;
    if(v < 0) {
        const char *e = getenv("SAGA_HIP_FORCE_DIRECT");
        v = (e && *e && *e != '0') ? 1 : 0;
    }
    return v == 1;
}

} // namespace

extern "C" {

size_t saga_hip_conv2d_workspace_size(int kind, const SagaTensorView *x, const SagaTensorView *w,
                                      const SagaTensorView *y, const SagaConvParams *p)
{
    ConvGeom g;
    if(geometry(x, w, y, p, &g))
        return 0;
    return std::max(conv_mfma_workspace(kind, x, w, y, g), conv_f32_workspace(kind, x, w, y, g));
}

// forward with the norm of `e` (+ residual + relu) in the epilogue
static int fwd_norm(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g,
                    const SagaConvExtras &e, void *workspace, size_t ws_bytes, hipStream_t st)
{
    if(force_direct())
        return SAGA_HIP_EUNSUPPORTED;
    if(x->dtype == SAGA_FLOAT) {
        if(e.z && (e.z->dtype != SAGA_FLOAT || !valid_view(e.z) || !same_dims(e.z, y)))
            return SAGA_HIP_EUNSUPPORTED;
        StreamEpilogue se;
        se.bn_s = e.s, se.bn_b = e.b, se.bn_m = e.m, se.bn_v = e.v;
        se.bn_eps = e.eps;
        se.z = e.z;
        se.relu = e.relu;
        return conv_f32_fwd(x, w, y, g, 1.0f, 0.0f, workspace, ws_bytes, st, se, e.packed);
    }
    const ConvBnFold bn = {e.s, e.b, e.m, e.v, e.eps, (e.z ? SAGA_BN_ADD : 0) | (e.relu ? SAGA_BN_RELU : 0), e.z};
    return conv_mfma_fwd(x, w, y, g, 1.0f, 0.0f, workspace, ws_bytes, st, nullptr, 0, nullptr, &bn, nullptr, nullptr, e.packed);
}

// whether backward data reads a filter that was transposed (fp16) or packed (fp32) beforehand
static bool takes_wt(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx, const ConvGeom &g)
{
    return !force_direct() && (dx->dtype == SAGA_FLOAT ? conv_f32_packed_bytes(SAGA_CONV_BWD_DATA, dx, w, dy, g) > 0
                                                       : conv_mfma_bwd_data_ok(dy, w, dx, g));
}

int saga_hip_conv2d_fwd(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                        const SagaConvParams *p, float alpha, float beta, void *workspace, size_t ws_bytes,
                        saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(!force_direct()) {
        r = conv_mfma_fwd(x, w, y, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
        r = conv_f32_fwd(x, w, y, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
    }
    return conv_direct_fwd(x, w, y, g, alpha, beta, as_stream(stream));
}

// the bias of a convolution into `out`, where no kernel takes it along
static int add_bias(const SagaTensorView *bias, const SagaTensorView *out, int relu, saga_stream_t stream)
{
    const int r = saga_hip_bias_add(out, bias, stream);
    return r || !relu ? r : saga_hip_act_fwd(SAGA_ACT_RELU, 0, out, out, 0.0f, stream);
}

static int check_bias(const SagaTensorView *bias, const SagaTensorView *out)
{
    int64_t step;
    if(!valid_view(bias) || view_elements(bias) != out->dims[1])
        return SAGA_HIP_ESHAPE;
    return as_vector(bias, &step) ? 0 : SAGA_HIP_EUNSUPPORTED;
}

// whether a kernel's epilogue can read it, which takes elements of this type next to each other
static bool fuses(const SagaTensorView *bias, int dtype)
{
    int64_t step;
    return bias && bias->dtype == dtype && as_vector(bias, &step) && step == 1;
}

int saga_hip_conv2d_fwd_ex(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                           float beta, const SagaConvExtras *e, void *workspace, size_t ws_bytes, saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(!e)
        return SAGA_HIP_EINVAL;
    hipStream_t st = as_stream(stream);
    if(e->s) {
        if(!e->b || !e->m || !e->v || e->bias || beta != 0.0f)
            return SAGA_HIP_EINVAL;
        return fwd_norm(x, w, y, g, *e, workspace, ws_bytes, st);
    }
    if(e->z || (e->relu && !e->bias))
        return SAGA_HIP_EUNSUPPORTED;
    const SagaTensorView *bias = e->bias;
    if(bias && (r = check_bias(bias, y)))
        return r;
    bool done = false;
    r = SAGA_HIP_EUNSUPPORTED;
    if(!force_direct()) {
        r = conv_mfma_fwd(x, w, y, g, 1.0f, beta, workspace, ws_bytes, st, nullptr, 0, nullptr, nullptr,
                          fuses(bias, SAGA_HALF) && !e->relu ? bias->ptr : nullptr, &done, e->packed);
        if(r == SAGA_HIP_EUNSUPPORTED) {
            StreamEpilogue se;
            done = fuses(bias, SAGA_FLOAT);
            if(done) {
                se.bias = (const float *)bias->ptr;
                se.relu = e->relu;
            }
            r = conv_f32_fwd(x, w, y, g, 1.0f, beta, workspace, ws_bytes, st, se, e->packed);
        }
    }
    if(r == SAGA_HIP_EUNSUPPORTED) {
        done = false;
        r = conv_direct_fwd(x, w, y, g, 1.0f, beta, st);
    }
    return r || done || !bias ? r : add_bias(bias, y, e->relu, stream);
}

size_t saga_hip_conv2d_pack_bytes(int kind, const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                                  const SagaConvParams *p)
{
    ConvGeom g;
    if(geometry(x, w, y, p, &g) || force_direct() || (kind != SAGA_CONV_FWD && kind != SAGA_CONV_BWD_DATA))
        return 0;
    if(x->dtype == SAGA_HALF)
        return kind == SAGA_CONV_FWD ? conv_mfma_packed_bytes(x, w, y, g) : 0;
    return conv_f32_packed_bytes(kind, x, w, y, g);
}

int saga_hip_conv2d_pack_jobs(int kind, const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                              const SagaConvParams *p, void *packed, SagaFilterPackJob *jobs)
{
    ConvGeom g;
    if(!packed || !jobs || !aligned16(packed) || !saga_hip_conv2d_pack_bytes(kind, x, w, y, p) || geometry(x, w, y, p, &g))
        return 0;
    if(x->dtype == SAGA_HALF) {
        conv_mfma_pack_job(w, g, packed, jobs[0]);
        return 1;
    }
    return stream_f32_pack_jobs(kind == SAGA_CONV_BWD_DATA, w, g, packed, jobs);
}

int saga_hip_filter_pack_batched(const SagaFilterPackJob *jobs_device, int njobs, int total_blocks, saga_stream_t stream)
{
    if(!jobs_device || njobs < 1 || total_blocks < 1)
        return SAGA_HIP_EINVAL;
    return stream_f32_pack(jobs_device, njobs, total_blocks, as_stream(stream));
}

int saga_hip_conv2d_bwd_data_bias(const SagaTensorView *dy, const SagaTensorView *w, const void *wt, const SagaTensorView *bias,
                                  const SagaTensorView *dx, const SagaConvParams *p, float beta, void *workspace, size_t ws_bytes,
                                  saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(dx, w, dy, p, &g);
    if(r)
        return r;
    if(bias && (r = check_bias(bias, dx)))
        return r;
    if(wt && !takes_wt(dy, w, dx, g))
        return SAGA_HIP_EUNSUPPORTED;
    hipStream_t st = as_stream(stream);
    bool done = false;
    r = SAGA_HIP_EUNSUPPORTED;
    if(!force_direct()) {
        r = conv_mfma_bwd_data(dy, w, dx, g, 1.0f, beta, workspace, ws_bytes, st, wt, nullptr,
                               fuses(bias, SAGA_HALF) ? bias->ptr : nullptr, &done);
        if(r == SAGA_HIP_EUNSUPPORTED) {
            StreamEpilogue e;
            done = fuses(bias, SAGA_FLOAT);
            if(done)
                e.bias = (const float *)bias->ptr;
            r = conv_f32_bwd_data(dy, w, dx, g, 1.0f, beta, workspace, ws_bytes, st, e, wt);
        }
    }
    if(r == SAGA_HIP_EUNSUPPORTED) {
        done = false;
        r = conv_direct_bwd_data(dy, w, dx, g, 1.0f, beta, st);
    }
    return r || done || !bias ? r : add_bias(bias, dx, 0, stream);
}

size_t saga_hip_conv2d_fwd_bnstats_size(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                                        const SagaConvParams *p)
{
    ConvGeom g;
    if(geometry(x, w, y, p, &g) || x->dtype != SAGA_HALF || force_direct())
        return 0;
    return conv_mfma_stats_floats(g) * sizeof(float);
}

int saga_hip_conv2d_fwd_bnstats(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                                const SagaConvParams *p, float alpha, void *workspace, size_t ws_bytes,
                                float *partial, size_t partial_bytes, int *partial_rows, saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(!partial || !partial_rows)
        return SAGA_HIP_EINVAL;
    if(force_direct())
        return SAGA_HIP_EUNSUPPORTED;
    return conv_mfma_fwd(x, w, y, g, alpha, 0.0f, workspace, ws_bytes, as_stream(stream), partial,
                         partial_bytes / sizeof(float), partial_rows);
}

int saga_hip_conv2d_fwd_bn_infer(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                                 const SagaTensorView *z, const SagaConvParams *p, const float *s, const float *b,
                                 const float *m, const float *v, float eps, int flags, void *workspace,
                                 size_t ws_bytes, saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(!s || !b || !m || !v || ((flags & SAGA_BN_ADD) && !z))
        return SAGA_HIP_EINVAL;
    const SagaConvExtras e = {nullptr, nullptr, s, b, m, v, eps, flags & SAGA_BN_ADD ? z : nullptr, flags & SAGA_BN_RELU ? 1 : 0};
    return fwd_norm(x, w, y, g, e, workspace, ws_bytes, as_stream(stream));
}

// geometry() of a convolution whose output there is no view of
static int pooled_geometry(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p, ConvGeom *g)
{
    if(!valid_view(x) || !valid_view(w) || !valid_view(y) || !p || p->stride < 1 || p->pad < 0 || p->dilation < 1)
        return SAGA_HIP_EINVAL;
    SagaTensorView between = *y;
    between.dims[1] = w->dims[0];
    between.dims[2] = conv_dim(x->dims[2], w->dims[2], p->pad, p->stride, p->dilation);
    between.dims[3] = conv_dim(x->dims[3], w->dims[3], p->pad, p->stride, p->dilation);
    return between.dims[2] < 1 || between.dims[3] < 1 ? SAGA_HIP_ESHAPE : geometry(x, w, &between, p, g);
}

int saga_hip_conv2d_fwd_bn_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                                      int pool_size, int pool_pad, int pool_stride)
{
    ConvGeom g;
    return !force_direct() && !pooled_geometry(x, w, y, p, &g) && conv_bn_maxpool_ok(x, w, y, g, pool_size, pool_pad, pool_stride);
}

int saga_hip_conv2d_fwd_bn_maxpool(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                                   const float *s, const float *b, const float *m, const float *v, float eps, int pool_size,
                                   int pool_pad, int pool_stride, saga_stream_t stream)
{
    ConvGeom g;
    const int r = pooled_geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(!s || !b || !m || !v)
        return SAGA_HIP_EINVAL;
    if(force_direct())
        return SAGA_HIP_EUNSUPPORTED;
    return conv_bn_maxpool(x, w, y, g, s, b, m, v, eps, pool_size, pool_pad, pool_stride, as_stream(stream));
}

// what follows the convolution, for a kernel that does a max pooling behind it; false: not that
static bool pooled_epilogue(const SagaTensorView *y, const SagaConvExtras *e, StreamEpilogue *se)
{
    if(!e || e->z || (e->s && (!e->b || !e->m || !e->v || e->bias)) || (e->bias && (check_bias(e->bias, y) || !fuses(e->bias, SAGA_FLOAT))))
        return false;
    se->bias = e->bias ? (const float *)e->bias->ptr : nullptr;
    se->bn_s = e->s, se->bn_b = e->b, se->bn_m = e->m, se->bn_v = e->v;
    se->bn_eps = e->eps;
    se->relu = e->relu;
    return true;
}

static bool pools_twos(const SagaTensorView *y, const ConvGeom &g, int size, int pad, int stride)
{
    return size == 2 && pad == 0 && stride == 2 && y->dims[0] == g.N && y->dims[1] == g.K && y->dims[2] == g.P / 2 && y->dims[3] == g.Q / 2;
}

int saga_hip_conv2d_fwd_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                                   const SagaConvExtras *e, int pool_size, int pool_pad, int pool_stride)
{
    ConvGeom g;
    StreamEpilogue se;
    return !force_direct() && !pooled_geometry(x, w, y, p, &g) && pools_twos(y, g, pool_size, pool_pad, pool_stride) &&
           pooled_epilogue(y, e, &se) && conv_f32_maxpool_ok(x, w, y, g, e->packed != nullptr);
}

int saga_hip_conv2d_fwd_maxpool(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const SagaConvParams *p,
                                const SagaConvExtras *e, int pool_size, int pool_pad, int pool_stride, void *workspace, size_t ws_bytes,
                                saga_stream_t stream)
{
    ConvGeom g;
    StreamEpilogue se;
    const int r = pooled_geometry(x, w, y, p, &g);
    if(r)
        return r;
    if(force_direct() || !pools_twos(y, g, pool_size, pool_pad, pool_stride) || !pooled_epilogue(y, e, &se))
        return SAGA_HIP_EUNSUPPORTED;
    return conv_f32_maxpool(x, w, y, g, workspace, ws_bytes, se, e->packed, as_stream(stream));
}

int saga_hip_conv2d_bwd_data(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx,
                             const SagaConvParams *p, float alpha, float beta, void *workspace, size_t ws_bytes,
                             saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(dx, w, dy, p, &g);
    if(r)
        return r;
    if(!force_direct()) {
        r = conv_mfma_bwd_data(dy, w, dx, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
        r = conv_f32_bwd_data(dy, w, dx, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
    }
    return conv_direct_bwd_data(dy, w, dx, g, alpha, beta, as_stream(stream));
}

size_t saga_hip_conv2d_bwd_data_wt_bytes(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx,
                                         const SagaConvParams *p)
{
    ConvGeom g;
    if(geometry(dx, w, dy, p, &g) || force_direct() || !conv_mfma_bwd_data_ok(dy, w, dx, g))
        return 0;
    return (size_t)g.K * g.C * g.R * g.S * 2;
}

int saga_hip_filter_transpose_blocks(const SagaTensorView *w)
{
    if(!valid_view(w))
        return 0;
    return conv_mfma_transpose_blocks(w->dims[0], w->dims[1], w->dims[2] * w->dims[3]);
}

int saga_hip_filter_transpose_batched(const SagaFilterTransposeJob *jobs_device, int njobs, int total_blocks,
                                      saga_stream_t stream)
{
    if(!jobs_device || njobs < 1 || total_blocks < 1)
        return SAGA_HIP_EINVAL;
    return conv_mfma_transpose_batched(jobs_device, njobs, total_blocks, as_stream(stream));
}

int saga_hip_conv2d_bwd_data_wt(const SagaTensorView *dy, const SagaTensorView *w, const void *wt, const SagaTensorView *dx,
                                const SagaConvParams *p, float alpha, float beta, void *workspace, size_t ws_bytes,
                                saga_stream_t stream)
{
    if(!wt)
        return saga_hip_conv2d_bwd_data(dy, w, dx, p, alpha, beta, workspace, ws_bytes, stream);
    ConvGeom g;
    int r = geometry(dx, w, dy, p, &g);
    if(r)
        return r;
    if(!takes_wt(dy, w, dx, g))
        return SAGA_HIP_EUNSUPPORTED;
    if(dx->dtype == SAGA_FLOAT)
        return conv_f32_bwd_data(dy, w, dx, g, alpha, beta, workspace, ws_bytes, as_stream(stream), StreamEpilogue(), wt);
    return conv_mfma_bwd_data(dy, w, dx, g, alpha, beta, workspace, ws_bytes, as_stream(stream), wt);
}

size_t saga_hip_conv2d_bwd_data_bnbwd_size(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx,
                                           const SagaConvParams *p)
{
    ConvGeom g;
    if(geometry(dx, w, dy, p, &g) || force_direct() || !conv_mfma_bnbwd_link_ok(dy, w, dx, g))
        return 0;
    return conv_mfma_bnbwd_floats(g) * sizeof(float);
}

int saga_hip_conv2d_bwd_data_bnbwd(const SagaTensorView *dy, const SagaTensorView *w, const void *wt,
                                   const SagaTensorView *dx, const SagaConvParams *p, float alpha, float beta,
                                   void *workspace, size_t ws_bytes, SagaBnBwdLink *link, saga_stream_t stream)
{
    if(!link || !valid_view(link->x) || !link->save_mean || !link->partial)
        return SAGA_HIP_EINVAL;
    if((link->flags & ~SAGA_BN_RELU) || ((link->flags & SAGA_BN_RELU) && (!link->s || !link->b || !link->save_invstd)))
        return SAGA_HIP_EINVAL;
    ConvGeom g;
    int r = geometry(dx, w, dy, p, &g);
    if(r)
        return r;
    if(force_direct() || !conv_mfma_bwd_data_ok(dy, w, dx, g))
        return SAGA_HIP_EUNSUPPORTED;
    int rows = 0;
    const ConvBnBwdLink l = {link->x, link->save_mean, link->save_invstd, link->s, link->b, link->flags & SAGA_BN_RELU,
                             link->partial, link->partial_bytes / sizeof(float), &rows};
    r = conv_mfma_bwd_data(dy, w, dx, g, alpha, beta, workspace, ws_bytes, as_stream(stream), wt, &l);
    if(r == 0)
        link->partial_rows = rows;
    return r;
}

int saga_hip_conv2d_bwd_filter(const SagaTensorView *x, const SagaTensorView *dy, const SagaTensorView *dw,
                               const SagaConvParams *p, float alpha, float beta, void *workspace,
                               size_t ws_bytes, saga_stream_t stream)
{
    ConvGeom g;
    int r = geometry(x, dw, dy, p, &g);
    if(r)
        return r;
    if(!force_direct()) {
        r = conv_mfma_bwd_filter(x, dy, dw, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
        r = conv_f32_bwd_filter(x, dy, dw, g, alpha, beta, workspace, ws_bytes, as_stream(stream));
        if(r != SAGA_HIP_EUNSUPPORTED)
            return r;
    }
    return conv_direct_bwd_filter(x, dy, dw, g, alpha, beta, as_stream(stream));
}

} // extern "C"
