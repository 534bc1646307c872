// One block of the network per call (sfno_block_*): the kernels of the filter, the norms, the MLP and the skip in the order
// makani/models/networks/sfnonet.py:239-267 applies them, enqueued from native code -- a dozen launches per direction without
// an interpreter between them -- and their backward.
#include <algorithm>
#include <cstdint>
#include <cstring>

#include "sfno_internal.h"

using namespace sfno;

namespace {

typedef unsigned short bf16;

// hands out 256-byte aligned pieces of a buffer; with a null base it only measures
struct Arena {
    char* base;
    size_t off = 0;
    explicit Arena(void* b) : base(reinterpret_cast<char*>(b)) {}
    int64_t take(size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) / 256 * 256;
        return (int64_t)at;
    }
    template <class T>
    T* get(size_t n) {
        const int64_t at = take(sizeof(T) * n);
        return reinterpret_cast<T*>(base + at);
    }
};

struct Dims {
    int B, ci, e, h, lmax, mmax, tri;
    int64_t P, Pin, rows_in, rows;            // pixels of the output and input grid; B * c_in, B * embed
    int64_t spec_in, spec_out, xm_in, xm_out; // floats
    bool scale_residual, one_mlp;
    bool valid = false;
    explicit Dims(const sfno_block* b) {
        if (!b || !b->fwd || !b->inv || b->batch < 1 || b->c_in < 1 || b->embed < 1 || b->hidden < 1) return;
        const sfno_sht_plan &f = *b->fwd, &i = *b->inv;
        if (f.lmax != i.lmax || f.mmax != i.mmax || (f.grid == SFNO_GRID_PLANAR) != (i.grid == SFNO_GRID_PLANAR)) return;
        B = b->batch; ci = b->c_in; e = b->embed; h = b->hidden;
        lmax = f.lmax; mmax = f.mmax; tri = f.grid == SFNO_GRID_PLANAR ? 0 : 1;
        P = (int64_t)i.nlat * i.nlon;
        Pin = (int64_t)f.nlat * f.nlon;
        if (P % 8 != 0) return;
        rows_in = (int64_t)B * ci;
        rows = (int64_t)B * e;
        scale_residual = f.nlat != i.nlat || f.nlon != i.nlon || f.grid != i.grid;
        spec_in = (int64_t)mmax * lmax * sfno_spectral_ld(rows_in);
        spec_out = (int64_t)mmax * lmax * sfno_spectral_ld(rows);
        xm_in = (int64_t)mmax * f.nlat * sfno_spectral_ld(rows_in);
        xm_out = (int64_t)mmax * i.nlat * sfno_spectral_ld(std::max(rows_in, rows));
        one_mlp = pointwise_mlp_preferred(B, e, h, P);
        valid = true;
    }
};

size_t layout(const Dims& d, bool training, int64_t off[SFNO_BLOCK_TENSORS]) {
    Arena a(nullptr);
    const size_t act = sizeof(bf16) * (size_t)d.rows * d.P, hid = sizeof(bf16) * (size_t)d.B * d.h * d.P;
    // inference: the coefficients are spent (residual and channel mix) when the filter's output is stored
    off[SFNO_BLOCK_SPEC] = a.take(std::max(sizeof(float) * (size_t)d.spec_in, training ? 0 : act));
    off[SFNO_BLOCK_X] = training ? a.take(act) : off[SFNO_BLOCK_SPEC];
    off[SFNO_BLOCK_COEF0] = training ? a.take(sizeof(float) * 4 * (size_t)d.rows) : -1;
    off[SFNO_BLOCK_H0] = training ? a.take(act) : off[SFNO_BLOCK_X];       // inference: norm0, GELU and MLP in place
    off[SFNO_BLOCK_Z1] = training ? a.take(hid) : -1;
    off[SFNO_BLOCK_A1] = training ? a.take(hid) : -1;                      // inference: in the workspace, over the filter's buffers
    off[SFNO_BLOCK_Y2] = training ? a.take(act) : off[SFNO_BLOCK_X];
    off[SFNO_BLOCK_COEF1] = a.take(sizeof(float) * 4 * (size_t)d.rows);
    off[SFNO_BLOCK_RES] = d.scale_residual ? a.take(sizeof(bf16) * (size_t)d.rows_in * d.P) : -1;
    return a.off;
}

// The buffers of a pass are laid over each other as far as their lifetimes allow.  Beside its state a training step of the full-size
// network with 4 layers then needs 14.0 GiB and a rollout of four samples with 8 layers 12.8; with buffers side by side 15.2 and 16.4.
struct FwdWs {
    float *xm_in, *xm_out, *spec, *coef0;
    float2 *stats, *partial;
    bf16* a1;                                            // null where norm0's GELU and the MLP are one kernel
    size_t bytes;
    FwdWs(const sfno_block* b, const Dims& d, void* base) {
        Arena a(base);
        coef0 = a.get<float>(4 * (size_t)d.rows);
        partial = a.get<float2>((size_t)d.rows * row_stats_segments(d.rows, d.P));
        Arena first = a, filter = a;
        xm_in = first.get<float>(d.xm_in);              // until the analysis
        spec = filter.get<float>(d.spec_out);           // from the channel mix until the synthesis
        xm_out = filter.get<float>(d.xm_out);
        stats = filter.get<float2>((size_t)d.rows * b->inv->nlat);
        a1 = d.one_mlp ? nullptr : a.get<bf16>((size_t)d.B * d.h * d.P);      // behind the filter
        bytes = std::max({a.off, first.off, filter.off});
    }
};

struct BwdWs {
    float *xm_in, *xm_out, *gspec_out, *gspec_in, *gspec_res, *wgrad_a, *wgrad_b;
    bf16 *dy2, *dz1, *dh0, *dx;
    float2* partial;
    size_t bytes, wgrad_bytes;
    BwdWs(const Dims& d, void* base) {
        Arena a(base);
        partial = a.get<float2>((size_t)d.rows * row_stats_segments(d.rows, d.P));
        wgrad_bytes = std::max({pointwise_wgrad_workspace_bytes(d.e, d.ci, 0, d.B, d.P), pointwise_wgrad_workspace_bytes(d.e, d.h, 1, d.B, d.P),
                                pointwise_wgrad_workspace_bytes(d.h, d.e, 1, d.B, d.P)});
        // two buffers in turn: dy2 -> dz1 -> dh0 -> dx, the shares of a weight gradient in the one whose tensor is not there yet or
        // spent; the filter's buffers over what is left of them behind dx, the last transform's over dx too
        const size_t at = a.off, dx_bytes = sizeof(bf16) * (size_t)std::max(d.rows, d.scale_residual ? d.rows_in : 0) * (size_t)d.P;
        dz1 = a.get<bf16>(std::max({sizeof(bf16) * (size_t)d.B * d.h * (size_t)d.P, dx_bytes, wgrad_bytes}) / sizeof(bf16));
        dy2 = a.get<bf16>(std::max(sizeof(bf16) * (size_t)d.rows * (size_t)d.P, wgrad_bytes) / sizeof(bf16));
        dx = dz1;
        dh0 = dy2;
        wgrad_a = reinterpret_cast<float*>(dz1);
        wgrad_b = reinterpret_cast<float*>(dy2);
        Arena filter = a;
        filter.off = at;
        filter.take(dx_bytes);
        xm_out = filter.get<float>(d.xm_out);
        gspec_out = filter.get<float>(std::max(d.spec_out, d.scale_residual ? d.spec_in : 0));
        gspec_res = gspec_out;                            // (gspec_out is spent once the input's coefficients have their gradient)
        Arena last = filter;
        last.off = at;
        xm_in = last.get<float>(d.xm_in);
        filter.off = std::max(filter.off, last.off);
        gspec_in = filter.get<float>(d.spec_in);
        bytes = std::max(a.off, filter.off);
    }
};

int conv(const bf16* x, const void* w, const float* bias, bf16* y, int B, int K, int O, int64_t P, int act, const bf16* addend, const float* scale,
         const float* shift, bf16* z, int grad, hipStream_t s) {
    PointwiseArgs a;
    std::memset(&a, 0, sizeof(a));
    a.X = x;
    a.W = reinterpret_cast<const bf16*>(w);
    a.bias = bias;
    a.Y = y;
    a.Z = z;
    a.grad = grad;
    a.addend = addend;
    a.add_scale = scale;
    a.add_shift = shift;
    a.K = K; a.O = O; a.B = B; a.act = act; a.P = P;
    return pointwise_gemm_launch(a, s);
}

// the kernels load and store 16 bytes at a time
template <class... T>
bool aligned(const T*... p) {
    return ((reinterpret_cast<uintptr_t>(p) | ...) & 15) == 0;
}

bool weights_fit(const sfno_dhconv_weights* w, int in, int out, int lmax) { return w && w->I == in && w->O == out && w->L == lmax; }

// adj holds the adjoint of p in the given direction
bool adjoint_of(const sfno_sht_plan* adj, const sfno_sht_plan* p, int direction) {
    return adj && (adj->directions & direction) && adj->nlat == p->nlat && adj->nlon == p->nlon && adj->lmax == p->lmax && adj->mmax == p->mmax &&
           adj->grid == p->grid && adj->norm == p->norm && adj->csphase == p->csphase && adj->device == p->device;
}

bool bf16_io(const sfno_sht_plan* p) { return sfno_sht_io_dtype_supported(p, SFNO_DTYPE_BF16) && sfno_sht_lat_stats_supported(p); }

}  // namespace

extern "C" size_t sfno_block_layout(const sfno_block* b, int training, int64_t offsets[SFNO_BLOCK_TENSORS]) {
    const Dims d(b);
    return d.valid && offsets ? layout(d, training != 0, offsets) : 0;
}

extern "C" size_t sfno_block_workspace_bytes(const sfno_block* b, int backward) {
    const Dims d(b);
    if (!d.valid) return 0;
    return backward ? BwdWs(d, nullptr).bytes : FwdWs(b, d, nullptr).bytes;
}

#define TRY(call)                          \
    do {                                   \
        const int rc_ = (call);            \
        if (rc_ != SFNO_OK) return rc_;    \
    } while (0)

extern "C" int sfno_block_forward(const sfno_block* b, int training, const void* x, void* out, void* kept, size_t kept_bytes, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    const Dims d(b);
    if (!d.valid || !x || !kept || !workspace || !aligned(x, out, kept, workspace)) return SFNO_EINVAL;
    if (!(b->fwd->directions & SFNO_DIR_FORWARD) || !(b->inv->directions & SFNO_DIR_INVERSE)) return SFNO_EINVAL;
    if (!weights_fit(b->weights, d.ci, d.e, d.lmax) || !b->w1 || !b->w2 || (out && !b->wskip)) return SFNO_EINVAL;
    if (!bf16_io(b->fwd) || !bf16_io(b->inv)) return SFNO_EUNSUPPORTED;
    int64_t off[SFNO_BLOCK_TENSORS];
    if (kept_bytes < layout(d, training != 0, off)) return SFNO_EWORKSPACE;
    const FwdWs w(b, d, workspace);
    if (workspace_bytes < w.bytes) return SFNO_EWORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    char* k = reinterpret_cast<char*>(kept);
    float* spec = reinterpret_cast<float*>(k + off[SFNO_BLOCK_SPEC]);
    bf16 *xf = (bf16*)(k + off[SFNO_BLOCK_X]), *h0 = (bf16*)(k + off[SFNO_BLOCK_H0]), *y2 = (bf16*)(k + off[SFNO_BLOCK_Y2]);
    bf16 *z1 = training ? (bf16*)(k + off[SFNO_BLOCK_Z1]) : nullptr, *a1 = training ? (bf16*)(k + off[SFNO_BLOCK_A1]) : w.a1;
    float *c0 = training ? (float*)(k + off[SFNO_BLOCK_COEF0]) : w.coef0, *c1 = (float*)(k + off[SFNO_BLOCK_COEF1]);
    const bf16* res = reinterpret_cast<const bf16*>(x);

    TRY(analysis_launch(b->fwd, x, SFNO_DTYPE_BF16, nullptr, w.xm_in, spec, d.rows_in, s));
    if (d.scale_residual) {
        bf16* r = (bf16*)(k + off[SFNO_BLOCK_RES]);
        TRY(synthesis_launch(b->inv, spec, w.xm_out, r, SFNO_DTYPE_BF16, nullptr, d.rows_in, s));
        res = r;
    }
    TRY(sfno_dhconv_spectral(b->weights, spec, w.spec, d.B, d.mmax, d.tri, s));
    float2* m0 = reinterpret_cast<float2*>(c0 + 2 * d.rows);
    if (d.P <= NORM_SMALL_PIXELS) {
        TRY(synthesis_launch(b->inv, w.spec, w.xm_out, xf, SFNO_DTYPE_BF16, nullptr, d.rows, s));
        TRY(instance_norm_coeffs_launch(xf, b->gamma0, b->beta0, c0, c0 + d.rows, w.partial, d.rows, d.e, d.P, b->eps0, s, m0));
    } else {
        TRY(synthesis_launch(b->inv, w.spec, w.xm_out, xf, SFNO_DTYPE_BF16, w.stats, d.rows, s));
        TRY(instance_norm_coeffs_lat_launch(w.stats, b->gamma0, b->beta0, c0, c0 + d.rows, d.rows, d.e, b->inv->nlat, b->eps0, s, m0));
    }
    if (!training && d.one_mlp) {
        MlpArgs m;
        std::memset(&m, 0, sizeof(m));
        m.X = xf;
        m.scale = c0;
        m.shift = c0 + d.rows;
        m.W1 = reinterpret_cast<const bf16*>(b->w1);
        m.b1 = b->b1;
        m.W2 = reinterpret_cast<const bf16*>(b->w2);
        m.b2 = b->b2;
        m.Y = y2;
        m.B = d.B; m.E = d.e; m.H = d.h; m.P = d.P;
        TRY(pointwise_mlp_launch(m, s));
    } else {
        TRY(scale_shift_act_launch(xf, c0, c0 + d.rows, h0, d.rows, d.P, training ? ACT_GELU_TRAIN : SFNO_ACT_GELU, s));
        TRY(conv(h0, b->w1, b->b1, a1, d.B, d.e, d.h, d.P, SFNO_ACT_GELU, nullptr, nullptr, nullptr, z1, 0, s));
        TRY(conv(a1, b->w2, b->b2, y2, d.B, d.h, d.e, d.P, SFNO_ACT_NONE, nullptr, nullptr, nullptr, nullptr, 0, s));
    }
    TRY(instance_norm_coeffs_launch(y2, b->gamma1, b->beta1, c1, c1 + d.rows, w.partial, d.rows, d.e, d.P, b->eps1, s, reinterpret_cast<float2*>(c1 + 2 * d.rows)));
    if (!out) return SFNO_OK;
    return conv(res, b->wskip, nullptr, reinterpret_cast<bf16*>(out), d.B, d.ci, d.e, d.P, SFNO_ACT_NONE, y2, c1, c1 + d.rows, nullptr, 0, s);
}

extern "C" int sfno_block_backward(const sfno_block* b, const void* gv, const void* x, const void* kept, size_t kept_bytes, const sfno_block_grads* grads,
                                   void* workspace, size_t workspace_bytes, void* stream) {
    const Dims d(b);
    if (!d.valid || !gv || !x || !kept || !grads || !workspace || !aligned(gv, x, kept, grads->gx, workspace)) return SFNO_EINVAL;
    if (!adjoint_of(b->fwd_adj, b->fwd, SFNO_DIR_FORWARD_ADJOINT) || !adjoint_of(b->inv_adj, b->inv, SFNO_DIR_INVERSE_ADJOINT)) return SFNO_EINVAL;
    const bool need_in = grads->gx || grads->gfilter, need_h0 = need_in || grads->ggamma0 || grads->gbeta0;
    if (!b->w2t || (need_h0 && !b->w1t) || (grads->gb1 && !grads->gw1) || (grads->gb2 && !grads->gw2)) return SFNO_EINVAL;
    if (grads->gx && (!b->wskipt || !weights_fit(b->weights_adj, d.e, d.ci, d.lmax))) return SFNO_EINVAL;
    int64_t off[SFNO_BLOCK_TENSORS];
    if (kept_bytes < layout(d, true, off)) return SFNO_EWORKSPACE;     // (the buffer of an inference call is smaller)
    const BwdWs w(d, workspace);
    if (workspace_bytes < w.bytes) return SFNO_EWORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    const char* k = reinterpret_cast<const char*>(kept);
    const float* spec = reinterpret_cast<const float*>(k + off[SFNO_BLOCK_SPEC]);
    const bf16 *xf = (const bf16*)(k + off[SFNO_BLOCK_X]), *h0 = (const bf16*)(k + off[SFNO_BLOCK_H0]), *z1 = (const bf16*)(k + off[SFNO_BLOCK_Z1]),
               *a1 = (const bf16*)(k + off[SFNO_BLOCK_A1]), *y2 = (const bf16*)(k + off[SFNO_BLOCK_Y2]);
    const float *c0 = (const float*)(k + off[SFNO_BLOCK_COEF0]), *c1 = (const float*)(k + off[SFNO_BLOCK_COEF1]);
    const bf16* res = d.scale_residual ? (const bf16*)(k + off[SFNO_BLOCK_RES]) : reinterpret_cast<const bf16*>(x);
    const bf16* g = reinterpret_cast<const bf16*>(gv);

    if (grads->gwskip) TRY(pointwise_wgrad_launch(g, res, grads->gwskip, nullptr, d.B, d.ci, d.e, d.P, w.wgrad_a, w.wgrad_bytes, s));
    // norm1, W2
    TRY(norm_grad_launch(g, y2, c1, c1 + d.rows, reinterpret_cast<const float2*>(c1 + 2 * d.rows), w.partial, w.dy2, grads->ggamma1, grads->gbeta1, d.B, d.e, d.P,
                         SFNO_ACT_NONE, s));
    if (grads->gw2) TRY(pointwise_wgrad_launch(w.dy2, a1, grads->gw2, grads->gb2, d.B, d.h, d.e, d.P, w.wgrad_a, w.wgrad_bytes, s));
    // GELU, W1
    TRY(conv(w.dy2, b->w2t, nullptr, w.dz1, d.B, d.e, d.h, d.P, SFNO_ACT_NONE, z1, nullptr, nullptr, nullptr, 1, s));
    if (grads->gw1) TRY(pointwise_wgrad_launch(w.dz1, h0, grads->gw1, grads->gb1, d.B, d.e, d.h, d.P, w.wgrad_b, w.wgrad_bytes, s));
    if (!need_h0) return SFNO_OK;
    TRY(conv(w.dz1, b->w1t, nullptr, w.dh0, d.B, d.h, d.e, d.P, SFNO_ACT_NONE, nullptr, nullptr, nullptr, nullptr, 0, s));
    // GELU, norm0
    TRY(norm_grad_launch(w.dh0, xf, c0, c0 + d.rows, reinterpret_cast<const float2*>(c0 + 2 * d.rows), w.partial, w.dx, grads->ggamma0, grads->gbeta0, d.B, d.e, d.P,
                         SFNO_ACT_GELU, s));
    if (!need_in) return SFNO_OK;
    // filter
    TRY(synthesis_adjoint_launch(b->inv_adj, w.dx, SFNO_DTYPE_BF16, w.xm_out, w.gspec_out, d.rows, s));
    if (grads->gfilter) {
        DhconvWgradArgs a;
        a.X = spec;
        a.G = w.gspec_out;
        a.GW = reinterpret_cast<float*>(grads->gfilter);
        a.B = d.B; a.I = d.ci; a.O = d.e; a.L = d.lmax; a.M = d.mmax;
        a.tri = d.tri;
        a.ld_in = (int)sfno_spectral_ld(d.rows_in);
        a.ld_out = (int)sfno_spectral_ld(d.rows);
        TRY(dhconv_wgrad_launch(a, s));
    }
    if (!grads->gx) return SFNO_OK;
    TRY(sfno_dhconv_spectral(b->weights_adj, w.gspec_out, w.gspec_in, d.B, d.mmax, d.tri, s));
    bf16* gx = reinterpret_cast<bf16*>(grads->gx);
    if (d.scale_residual) {
        // the residual's gradient joins in spectral space
        TRY(conv(g, b->wskipt, nullptr, w.dx, d.B, d.e, d.ci, d.P, SFNO_ACT_NONE, nullptr, nullptr, nullptr, nullptr, 0, s));
        TRY(synthesis_adjoint_launch(b->inv_adj, w.dx, SFNO_DTYPE_BF16, w.xm_out, w.gspec_res, d.rows_in, s));
        TRY(spectral_add_launch(w.gspec_in, w.gspec_res, d.lmax, d.mmax, (int)sfno_spectral_ld(d.rows_in), d.tri, s));
        return analysis_adjoint_launch(b->fwd_adj, w.gspec_in, gx, SFNO_DTYPE_BF16, w.xm_in, d.rows_in, s);
    }
    TRY(analysis_adjoint_launch(b->fwd_adj, w.gspec_in, gx, SFNO_DTYPE_BF16, w.xm_in, d.rows_in, s));
    // skip gradient on top, in place
    return conv(g, b->wskipt, nullptr, gx, d.B, d.e, d.ci, d.P, SFNO_ACT_NONE, gx, nullptr, nullptr, nullptr, 0, s);
}
