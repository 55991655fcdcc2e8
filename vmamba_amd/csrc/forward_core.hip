// forward_core of a one-state block as one call (classification/models/vmamba.py:603-646): x_proj, dt_proj, the fused core and
// out_norm enqueued back to back.  The kernels are those of the separate entry points -- but for large maps of few ranks, where
// dt_proj is folded into the core --; what this saves is the host's share.
// From Python the four launches, their argument checks, tensors and views took 81 us for one map of 768 x 7 x 7 whose kernels
// run for 38 -- and most of a 15-block model's time on one image.  One call with one workspace takes the host's share out of
// everything but the largest batches.
#include "scan_common.h"

namespace ss2d {

struct ForwardCorePlan {
    bool padded, few;                                                // few: core_few.hip's two kernels
    DtsLayout layout;
    int planes, flags_per_image;                                     // planes > 0: dt_proj folded into the core
    int64_t pitch, x, x_dbl, flags, delta, y, out, scratch, total;   // row pitch in elements; byte offsets; bytes
    ss2d_core_params core;
};

// What a kernel refuses is found here, before a caller has allocated or launched anything.
static bool forward_core_kernels_take(const ss2d_forward_core_params *q, int64_t pitch) {
    if (q->dtype == SS2D_F32) {
        if (!dt_proj_f32_takes(q->rank)) return false;
    } else if (ss2d_x_proj_applies(q->batch, q->dim, q->rank + 2, q->padded_height, q->padded_width, q->dtype) != SS2D_OK ||
               reinterpret_cast<uintptr_t>(q->x_proj_weight) % 16 != 0 || !dt_proj_takes(q->dim, q->rank, pitch, pitch, q->dtype)) {
        return false;
    }
    return !q->normalise || layer_norm_cf_takes(q->dim, SS2D_F32, q->norm_dtype, q->dtype);
}

// Elements of the map from which dt_proj is folded into the core where the core takes that (core_dts_takes): 96 x 56 x 56, batch 128,
// bf16 292 -> 234 us, 64 x 96 x 96, batch 33 225 -> 177, 48 x 96 maps of 57 x 58, fp16 159 -> 150, 54 x 128 x 8 x 9 (0.5 Mi elements)
// 26 -> 22.  Below it a call is bound by its launches and the host, there is less to win (0.1 Mi elements, in a graph: 18.4 -> 16.2),
// and small calls keep the bits of the kernels one by one.  The line is one of rounding too: above it the step is the fp32 sum over its
// ranks, below it that sum rounded to 16 bits, so an image alone and the same image in a large batch differ by that rounding.
constexpr int64_t kFoldFrom = 1 << 19;

static int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// base may be NULL while only the size is asked for: stand-in pointers of the same alignment take its place
static int forward_core_plan(const ss2d_forward_core_params *q, char *base, ForwardCorePlan &p) {
    if (!q) return SS2D_EINVAL;
    if (q->batch <= 0 || q->dim <= 0 || q->height <= 0 || q->width <= 0 || q->rank <= 0) return SS2D_EINVAL;
    if (q->dtype != SS2D_F32 && q->dtype != SS2D_BF16 && q->dtype != SS2D_F16) return SS2D_EINVAL;
    if (!q->x || !q->x_proj_weight || !q->dt_proj_weight || !q->A || !q->out) return SS2D_EINVAL;
    if (q->padded_height < q->height || q->padded_width < q->width) return SS2D_EINVAL;
    p.padded = q->padded_height > q->height || q->padded_width > q->width;
    if (p.padded && (q->dtype == SS2D_F32 || !q->pad_mask)) return q->dtype == SS2D_F32 ? SS2D_ENOTSUP : SS2D_EINVAL;
    const int64_t L = (int64_t)q->padded_height * q->padded_width, D = q->dim, C = q->rank + 2, es = q->dtype == SS2D_F32 ? 4 : 2;
    // rows of batch * L positions, kept on 16-byte boundaries: the next kernels then keep their vector accesses
    const int64_t vec = 16 / es;
    p.pitch = (q->batch * L + vec - 1) / vec * vec;
    // on a padded map delta has to start every image where its mask does
    if (p.padded && p.pitch != q->batch * L) return SS2D_ENOTSUP;
    p.few = !p.padded && few_pays(q->batch, q->dim, q->rank, q->height, q->width, q->dtype) && reinterpret_cast<uintptr_t>(q->x_proj_weight) % 16 == 0;
    if (p.few) {
        if (q->dtype == SS2D_F32 && !dt_proj_f32_takes(q->rank)) return SS2D_ENOTSUP;
        if (q->normalise && !layer_norm_cf_takes(q->dim, SS2D_F32, q->norm_dtype, q->dtype)) return SS2D_ENOTSUP;
        p.x_dbl = 0;
        p.y = align256(few_rows_bytes(q->batch, q->rank, L, q->dtype));
        p.total = align256(p.y + (q->normalise ? q->batch * D * L * 4 : 0));
        return SS2D_OK;
    }
    if (!forward_core_kernels_take(q, p.pitch)) return SS2D_ENOTSUP;
    p.x = 0;
    p.x_dbl = p.padded ? align256(p.x + q->batch * D * L * es) : 0;
    char *const at = base ? base : reinterpret_cast<char *>(256);
    ss2d_core_params &c = p.core;
    c.batch = q->batch; c.dim = q->dim; c.height = q->padded_height; c.width = q->padded_width;
    c.in_dtype = q->dtype; c.delta_softplus = 1;
    c.x = p.padded ? at + p.x : q->x; c.A = q->A; c.D = q->D; c.delta_bias = q->delta_bias;
    c.delta_dir_stride = D * p.pitch; c.delta_dim_stride = p.pitch; c.delta_batch_stride = L;
    c.B_batch_stride = c.C_batch_stride = L;
    auto rows = [&](int64_t n) {                                     // of x_proj per direction, the last two of them B and C
        c.B = at + p.x_dbl + (n - 2) * p.pitch * es; c.C = at + p.x_dbl + (n - 1) * p.pitch * es;
        c.B_dir_stride = c.C_dir_stride = n * p.pitch;
        p.flags = align256(p.x_dbl + 4 * n * p.pitch * es);
    };
    c.delta = c.y = at;                                              // (until their places are known)
    p.planes = 0;
    if (q->dtype != SS2D_F32 && q->batch * D * L >= kFoldFrom) {
        const int planes = dts_planes(q->rank, p.padded);
        rows(2 * planes + 2);
        p.flags_per_image = x_proj_pairs_workgroups(q->batch, q->dim, q->rank, q->padded_height, q->padded_width, q->dtype);
        if (p.flags_per_image > 0 && core_dts_takes(&c, q->rank, p.padded, (planes + 1) * p.pitch, p.pitch, p.layout)) p.planes = planes;
    }
    if (p.planes > 0) {
        p.delta = align256(p.flags + (int64_t)q->batch * p.flags_per_image * 4);
        p.y = align256(p.delta + (q->normalise && p.padded ? q->batch * D * L * es : 0));      // (no delta: the normalised padded map alone)
    } else {
        rows(C);
        p.delta = p.flags;
        p.y = align256(p.delta + 4 * D * p.pitch * es);
    }
    p.out = p.delta;                                                 // the normalised padded map: four times its room, and read already
    p.scratch = q->normalise || p.padded ? align256(p.y + q->batch * D * L * 4) : p.y;
    c.delta = at + p.delta;
    c.y = q->normalise || p.padded ? at + p.y : q->out;
    const int64_t need = ss2d_core_workspace_bytes(&c);
    if (need < 0) return (int)need;
    p.total = align256(p.scratch + need);
    return SS2D_OK;
}

}  // namespace ss2d

extern "C" int64_t ss2d_forward_core_workspace_bytes(const ss2d_forward_core_params *q) {
    ss2d::ForwardCorePlan p;
    const int rc = ss2d::forward_core_plan(q, nullptr, p);
    return rc != SS2D_OK ? rc : p.total;
}

extern "C" int ss2d_forward_core(const ss2d_forward_core_params *q, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return SS2D_EINVAL;
    ForwardCorePlan p;
    char *const base = reinterpret_cast<char *>(workspace);
    int rc = forward_core_plan(q, base, p);
    if (rc != SS2D_OK) return rc;
    if (workspace_bytes < p.total) return SS2D_ENOMEM;
    const int B = q->batch, D = q->dim, H = q->padded_height, W = q->padded_width, R = q->rank, C = R + 2;
    const int64_t L = (int64_t)H * W, ks = C * p.pitch;
    const int es = q->dtype == SS2D_F32 ? 4 : 2;
    if (p.few) {
        float *y = q->normalise ? (float *)(base + p.y) : (float *)q->out;
        rc = ss2d_x_proj_few(q->x, q->x_proj_weight, base + p.x_dbl, B, D, R, H, W, q->dtype, stream);
        if (rc == SS2D_OK) rc = ss2d_core_few(q->x, base + p.x_dbl, q->dt_proj_weight, (const float *)q->A, (const float *)q->D, (const float *)q->delta_bias, y, B, D, R, H, W, q->dtype, stream);
        if (rc == SS2D_OK && q->normalise)
            rc = ss2d_layer_norm_cf(y, q->norm_weight, q->norm_bias, q->out, B, D, (int)L, q->eps, SS2D_F32, q->norm_dtype, q->dtype, q->out_channel_last, stream);
        return rc;
    }
    void *x_dbl = base + p.x_dbl, *delta = base + p.delta;
    if (p.padded) rc = ss2d_core_embed_maps(q->x, base + p.x, (int64_t)B * D, q->height, q->width, H, W, es, stream);
    const void *x = p.core.x;
    if (p.planes > 0) {
        // a step of softplus(fill) = 0 at the added positions, through a rank of their own
        const int64_t rows = 2 * p.planes + 2;
        if (rc == SS2D_OK) rc = x_proj_pairs(x, q->x_proj_weight, x_dbl, (int32_t *)(base + p.flags), B, D, R, H, W, q->height, q->width, rows * p.pitch,
                                             p.pitch, p.layout, q->dtype, stream);
        const CoreDts t = {x_dbl, q->dt_proj_weight, rows * p.pitch / 2, p.pitch, R, !p.padded ? 0u : q->dtype == SS2D_F16 ? 0xfbffu : 0xf149u,
                           (const int32_t *)(base + p.flags), p.flags_per_image};
        if (rc == SS2D_OK) rc = core_dts_fwd(&p.core, t, (hipStream_t)stream);
    } else if (q->dtype == SS2D_F32) {
        rc = ss2d_x_proj_f32((const float *)x, (const float *)q->x_proj_weight, (float *)x_dbl, B, D, C, H, W, ks, p.pitch, L, stream);
        if (rc == SS2D_OK) rc = ss2d_dt_proj_f32((const float *)x_dbl, (const float *)q->dt_proj_weight, (float *)delta, 4, D, R, p.pitch, ks, p.pitch, stream);
    } else {
        if (rc == SS2D_OK) rc = ss2d_x_proj(x, q->x_proj_weight, x_dbl, B, D, C, H, W, H, W, -1, ks, p.pitch, L, q->dtype, stream);
        // a step of softplus(fill) = 0 at the added positions
        if (rc == SS2D_OK) rc = ss2d_dt_proj_masked(x_dbl, q->dt_proj_weight, p.padded ? q->pad_mask : nullptr, q->dtype == SS2D_F16 ? -65504.0f : -1e30f,
                                                    delta, 4, D, R, p.pitch, ks, p.pitch, q->dtype, stream);
    }
    if (rc == SS2D_OK && p.planes == 0) rc = ss2d_core_fwd_ws(&p.core, base + p.scratch, p.total - p.scratch, stream);
    if (rc == SS2D_OK && q->normalise && p.padded && q->out_channel_last) {
        rc = ss2d_layer_norm_cf_crop((const float *)(base + p.y), q->norm_weight, q->norm_bias, q->out, B, D, H, W, q->height, q->width, q->eps,
                                     q->norm_dtype, q->dtype, stream);
        if (rc != SS2D_ENOTSUP) return rc;
        rc = SS2D_OK;
    }
    if (rc == SS2D_OK && q->normalise)
        rc = ss2d_layer_norm_cf(base + p.y, q->norm_weight, q->norm_bias, p.padded ? base + p.out : q->out, B, D, (int)L, q->eps, SS2D_F32,
                                q->norm_dtype, q->dtype, q->out_channel_last, stream);
    if (rc != SS2D_OK || !p.padded) return rc;
    if (!q->normalise) return ss2d_core_embed_maps(base + p.y, q->out, (int64_t)B * D, H, W, q->height, q->width, 4, stream);
    if (q->out_channel_last)                                         // an image is one map of H rows of W * D elements
        return ss2d_core_embed_maps(base + p.out, q->out, B, H, (int64_t)W * D, q->height, (int64_t)q->width * D, es, stream);
    return ss2d_core_embed_maps(base + p.out, q->out, (int64_t)B * D, H, W, q->height, q->width, es, stream);
}
