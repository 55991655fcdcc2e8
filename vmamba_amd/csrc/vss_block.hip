// A block of few positions as one call (classification/models/vmamba.py:1225-1229): LayerNorm + in_proj, the depthwise convolution,
// forward_core, out_proj + add, and where the positions are few enough LayerNorm + fc1 + GELU and
// fc2 + add, enqueued back to back.  The kernels are those of the separate
// entry points and so are the results; what this saves is the host's share: six calls with their checks, tensors and views took
// 100-120 us a block from Python, on one image twice the time of the kernels.
#include "ss2d_common.h"

namespace ss2d {

struct BlockPlan {
    ss2d_forward_core_params core;
    bool mlp;                                                        // fc1 and fc2 are there
    bool narrow;                                                     // out_norm + out_proj + add in one kernel (ss2d_linear_cf_ln)
    int64_t proj, conv, mixed, sum, hidden, core_ws, core_bytes, total;   // byte offsets in the workspace; bytes
};

// What a kernel of the block refuses is found here, before a caller has allocated or launched anything.
static bool block_kernels_take(const ss2d_block_params *q, int64_t M) {
    const int C = q->d_model, D = q->core.dim, hidden = q->hidden, dt = q->core.dtype;
    const void *const ptrs[] = {q->x, q->residual, q->norm_weight, q->norm_bias, q->in_proj_weight, q->in_proj_bias, q->core.norm_weight, q->core.norm_bias,
                                q->out_proj_weight, q->out_proj_bias, q->norm2_weight, q->norm2_bias, q->fc1_weight, q->fc1_bias, q->fc2_weight,
                                q->fc2_bias, q->out};
    for (const void *at : ptrs)
        if (reinterpret_cast<uintptr_t>(at) % 16 != 0) return false;
    if ((int64_t)q->core.height * q->core.width > 0x3fffffff) return false;                       // the convolution's
    return linear_rows_takes(M, C, D, q->norm_weight != nullptr, dt) && linear_rows_takes(M, D, C, false, dt) &&
           (!q->fc1_weight || (linear_rows_takes(M, C, hidden, true, dt) && linear_rows_takes(M, hidden, C, false, dt)));
}

static int block_plan(const ss2d_block_params *q, char *base, BlockPlan &p) {
    if (!q) return SS2D_EINVAL;
    p.core = q->core;
    if (p.core.dtype != SS2D_BF16 && p.core.dtype != SS2D_F16) return p.core.dtype == SS2D_F32 ? SS2D_ENOTSUP : SS2D_EINVAL;
    if (p.core.batch <= 0 || p.core.height <= 0 || p.core.width <= 0 || p.core.dim <= 0 || q->d_model <= 0 || q->hidden <= 0) return SS2D_EINVAL;
    if (!q->x || !q->out || !q->in_proj_weight || !q->conv_weight || !q->out_proj_weight ||
        !p.core.norm_weight)
        return SS2D_EINVAL;
    p.mlp = q->fc1_weight != nullptr;
    if (p.mlp && (!q->fc2_weight || !q->norm2_weight)) return SS2D_EINVAL;
    if (!q->norm_weight && !q->residual) return SS2D_EINVAL;         // (a normalised x is not the residual stream)
    if (q->norm_bias && !q->norm_weight) return SS2D_EINVAL;
    const int64_t M = (int64_t)p.core.batch * p.core.height * p.core.width, D = p.core.dim;
    if (!block_kernels_take(q, M)) return SS2D_ENOTSUP;
    auto align = [](int64_t v) { return (v + 255) & ~(int64_t)255; };
    const int64_t L = (int64_t)p.core.height * p.core.width;
    p.narrow = q->d_model == 96 && D == 96 && L % 32 == 0 && p.core.norm_dtype == p.core.dtype;
    p.proj = 0;
    p.conv = align(p.proj + M * D * 2);
    p.mixed = align(p.conv + M * D * 2);
    p.sum = align(p.mixed + M * D * (p.narrow ? 4 : 2));
    p.hidden = align(p.sum + (p.mlp ? M * q->d_model * 2 : 0));
    p.core_ws = align(p.hidden + (p.mlp ? M * q->hidden * 2 : 0));
    char *const at = base ? base : reinterpret_cast<char *>(256);    // (only the size is asked for: stand-ins of the same alignment)
    p.core.x = at + p.conv;
    p.core.out = at + p.mixed;
    p.core.normalise = !p.narrow;
    p.core.out_channel_last = 1;
    p.core_bytes = ss2d_forward_core_workspace_bytes(&p.core);
    if (p.core_bytes < 0) return (int)p.core_bytes;
    p.total = p.core_ws + p.core_bytes;
    return SS2D_OK;
}

}  // namespace ss2d

extern "C" int64_t ss2d_block_workspace_bytes(const ss2d_block_params *q) {
    ss2d::BlockPlan p;
    const int rc = ss2d::block_plan(q, nullptr, p);
    return rc != SS2D_OK ? rc : p.total;
}

extern "C" int ss2d_block_fwd(const ss2d_block_params *q, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace ss2d;
    if (!workspace || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return SS2D_EINVAL;
    BlockPlan p;
    char *const base = reinterpret_cast<char *>(workspace);
    int rc = block_plan(q, base, p);
    if (rc != SS2D_OK) return rc;
    if (workspace_bytes < p.total) return SS2D_ENOMEM;
    const ss2d_forward_core_params &c = p.core;
    const int C = q->d_model, D = c.dim, dt = c.dtype;
    const int64_t M = (int64_t)c.batch * c.height * c.width;
    const void *residual = q->residual ? q->residual : q->x;
    void *sum = p.mlp ? base + p.sum : q->out;
    // 96 -> 96 of many positions: the kernel that holds the weights and walks over tiles.  bf16, in a graph, ss2d_linear_rows against it in
    // us: with the LayerNorm 12 544 positions 4.9 / 8.0, 25 088 7.0 / 8.3, 31 360 8.8 / 8.5, 43 904 10.9 / 8.9 (the line is the separate
    // calls', linear_rows_pays).  out_proj with its residual crosses later, 29 760 7.3 / 8.5, 37 632 9.0 / 9.4, 43 904 10.0 / 9.1, and in
    // the block, behind the norm that has just written its operand, no earlier than its most positions (two blocks of 8 x 60 x 62
    // 192 / 198, of 12 x 60 x 62 244 / 244): ss2d_linear_rows throughout.
    if (C == 96 && D == 96 && M > 24576)
        rc = ss2d_linear_cl(q->x, q->norm_weight, q->norm_bias, q->norm_eps, q->in_proj_weight, q->in_proj_bias, nullptr, base + p.proj, M, C, D, dt, stream);
    else
        rc = ss2d_linear_rows(q->x, q->norm_weight, q->norm_bias, q->norm_eps, q->in_proj_weight, q->in_proj_bias, nullptr, base + p.proj, M, C, D, 0, dt,
                              stream);
    if (rc == SS2D_OK) rc = ss2d_dwconv3x3_silu(base + p.proj, q->conv_weight, q->conv_bias, base + p.conv, c.batch, D, c.height, c.width, dt, 1, 1, stream);
    if (rc == SS2D_OK) rc = ss2d_forward_core(&p.core, base + p.core_ws, p.core_bytes, stream);
    if (rc == SS2D_OK && p.narrow)
        rc = ss2d_linear_cf_ln(base + p.mixed, c.norm_weight, c.norm_bias, c.eps, q->out_proj_weight, q->out_proj_bias, residual, sum, c.batch,
                               c.height * c.width, D, C, dt, stream);
    else if (rc == SS2D_OK)
        rc = ss2d_linear_rows(base + p.mixed, nullptr, nullptr, 0.0f, q->out_proj_weight, q->out_proj_bias, residual, sum, M, D, C, 0, dt, stream);
    if (rc != SS2D_OK || !p.mlp) return rc;
    rc = ss2d_linear_rows(base + p.sum, q->norm2_weight, q->norm2_bias, q->norm2_eps, q->fc1_weight, q->fc1_bias, nullptr, base + p.hidden, M, C,
                          q->hidden, 1, dt, stream);
    if (rc == SS2D_OK)
        rc = ss2d_linear_rows(base + p.hidden, nullptr, nullptr, 0.0f, q->fc2_weight, q->fc2_bias, base + p.sum, q->out, M, q->hidden, C, 0, dt, stream);
    return rc;
}
