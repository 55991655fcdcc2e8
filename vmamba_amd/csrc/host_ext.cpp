// The host's share of forward_core, of a block of few positions and of the three operators, in C++: the checks of their tensors, the outputs and
// workspaces and the calls into the C ABI.  Through ctypes and torch's Python interface that took 14 us of a forward_core whose three kernels
// run for 18, 20 us of a block, and most of what the three operators take on a few small maps (2 x 96 of 14 x 14: inference 38 us, so 24;
// forward and backward 161, 98; with 16 states forward_core 113, 75).  No kernel lives here, and what is checked is what the Python callers (core.py, block.py, csm.py, csms6s.py) checked.
#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <array>

#include "../../include/ss2d_hip.h"

namespace py = pybind11;

static int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::ScalarType::Float: return SS2D_F32;
        case at::ScalarType::BFloat16: return SS2D_BF16;
        case at::ScalarType::Half: return SS2D_F16;
        default: return -1;
    }
}

static const void *ptr_of(const at::Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
static bool has_shape(const at::Tensor &t, at::IntArrayRef sizes) { return t.sizes() == sizes; }
static bool on(const at::Tensor &t, const at::Tensor &x) { return t.is_cuda() && t.get_device() == x.get_device(); }
// a view with a conjugate or negative bit still to be applied is not its memory; neither is a tensor without any
static bool plain(const at::Tensor &t) { return !t.is_conj() && !t.is_neg() && t.has_storage() && t.layout() == at::kStrided; }

// fn() without Python's lock, on x's device and PyTorch's current stream there
template <typename F> static int enqueue(const at::Tensor &x, F fn) {
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    void *stream = (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    py::gil_scoped_release unlocked;
    return fn(stream);
}

// core.py:forward_core_hip -- the tensor, None where the kernels do not stand for the call, or the status of a failed one.
static py::object forward_core(const at::Tensor &x_in, const at::Tensor &x_proj, const at::Tensor &dt_proj, const at::Tensor &A, const at::Tensor &D,
                               const at::Tensor &dt_bias, const c10::optional<at::Tensor> &norm_weight, const c10::optional<at::Tensor> &norm_bias,
                               double eps, bool normalise, bool channel_last, int64_t padded_h, int64_t padded_w,
                               const c10::optional<at::Tensor> &pad_mask) {
    const int code = dtype_code(x_in.scalar_type());
    if (code < 0 || x_in.numel() == 0 || dt_proj.dim() != 3) return py::none();
    const int64_t B = x_in.size(0), Dm = x_in.size(1), H = x_in.size(2), W = x_in.size(3), R = dt_proj.size(2);
    if (R == 0 || !has_shape(x_proj, {4, R + 2, Dm}) || !has_shape(dt_proj, {4, Dm, R})) return py::none();
    for (const at::Tensor *t : {&x_proj, &dt_proj})
        if (t->scalar_type() != x_in.scalar_type() || !on(*t, x_in) || !t->is_contiguous() || !plain(*t)) return py::none();
    for (const at::Tensor *t : {&A, &D, &dt_bias})
        if (t->numel() != 4 * Dm || t->scalar_type() != at::ScalarType::Float || !on(*t, x_in) || !t->is_contiguous()) return py::none();
    const at::Tensor x = x_in.contiguous();
    ss2d_forward_core_params p = {};
    p.batch = (int)B; p.dim = (int)Dm; p.height = (int)H; p.width = (int)W; p.rank = (int)R;
    p.padded_height = (int)padded_h; p.padded_width = (int)padded_w; p.dtype = code;
    if (pad_mask.has_value()) p.pad_mask = pad_mask->data_ptr();
    at::Tensor out;
    if (normalise) {
        const at::Tensor w = norm_weight.value_or(at::Tensor()), b = norm_bias.value_or(at::Tensor());
        for (const at::Tensor *t : {&w, &b})
            if (t->defined() && (!on(*t, x) || !t->is_contiguous() || !plain(*t) || t->numel() != Dm || dtype_code(t->scalar_type()) < 0)) return py::none();
        if (w.defined() && b.defined() && w.scalar_type() != b.scalar_type()) return py::none();
        p.normalise = 1; p.out_channel_last = channel_last ? 1 : 0; p.eps = (float)eps;
        p.norm_weight = ptr_of(w); p.norm_bias = ptr_of(b);
        p.norm_dtype = w.defined() || b.defined() ? dtype_code((w.defined() ? w : b).scalar_type()) : SS2D_F32;
        out = channel_last ? at::empty({B, H, W, Dm}, x.options()) : at::empty({B, Dm, H, W}, x.options());
    } else {
        out = at::empty({B, Dm, H * W}, x.options().dtype(at::kFloat));
    }
    p.x = x.data_ptr(); p.x_proj_weight = x_proj.data_ptr(); p.dt_proj_weight = dt_proj.data_ptr();
    p.A = A.data_ptr(); p.D = D.data_ptr(); p.delta_bias = dt_bias.data_ptr(); p.out = out.data_ptr();
    const int64_t need = ss2d_forward_core_workspace_bytes(&p);
    if (need == SS2D_ENOTSUP) return py::none();
    if (need < 0) return py::int_(need);
    at::Tensor workspace = at::empty({need}, x.options().dtype(at::kByte));
    const int rc = enqueue(x, [&](void *stream) { return ss2d_forward_core(&p, workspace.data_ptr(), need, stream); });
    if (rc == SS2D_ENOTSUP) return py::none();
    return rc != SS2D_OK ? py::object(py::int_(rc)) : py::cast(out);
}

// The tensor behind an object of exactly one of `kinds`; undefined for None and, with ok = false, for anything else.
static at::Tensor exactly(const py::handle &h, const py::tuple &kinds, bool &ok) {
    if (h.is_none()) return {};
    for (const py::handle &kind : kinds)
        if ((PyObject *)Py_TYPE(h.ptr()) == kind.ptr()) return THPVariable_Unpack(h.ptr());
    ok = false;
    return {};
}

// block.py:vss_block_hip from its tensors on.  weights, biases: in_proj, out_proj, fc1, fc2, norm, norm2, out_norm, conv; eps: norm, norm2,
// out_norm; whole: with the MLP; kinds: the types whose memory is theirs.  The tensor, None where the call does not stand for
// the modules, or the status of a failed one.
static py::object block(const py::tuple &kinds, const py::object &x_in, const py::object &residual_in, const py::tuple &weights, const py::tuple &biases,
                        const py::object &x_proj_in, const py::object &dt_proj_in, const at::Tensor &A, const at::Tensor &D, const at::Tensor &dt_bias,
                        const std::array<double, 3> &eps, bool whole) {
    constexpr size_t kLayers = 8;
    if (weights.size() != kLayers || biases.size() != kLayers) throw std::invalid_argument("eight weights and eight biases");
    bool ok = true;
    const at::Tensor x = exactly(x_in, kinds, ok), residual = exactly(residual_in, kinds, ok);
    const at::Tensor x_proj = exactly(x_proj_in, kinds, ok), dt_proj = exactly(dt_proj_in, kinds, ok);
    if (!ok || !x.defined() || !x_proj.defined() || !dt_proj.defined() || x.dim() != 4 || dt_proj.dim() != 3) return py::none();
    const int code = dtype_code(x.scalar_type());
    if (code != SS2D_BF16 && code != SS2D_F16) return py::none();
    auto readable = [&](const at::Tensor &t) {
        return t.scalar_type() == x.scalar_type() && on(t, x) && plain(t) && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    };
    if (!readable(x) || !readable(x_proj) || !readable(dt_proj) || (residual.defined() && (!readable(residual) || residual.sizes() != x.sizes()))) return py::none();
    at::Tensor w[kLayers], b[kLayers];
    for (size_t i = 0; i < kLayers; ++i) {
        w[i] = exactly(weights[i], kinds, ok);
        b[i] = exactly(biases[i], kinds, ok);
        if (!ok || !w[i].defined() || !readable(w[i]) || (b[i].defined() && !readable(b[i]))) return py::none();
    }
    enum { kIn, kOut, kFc1, kFc2, kNorm, kNorm2, kOutNorm, kConv };
    const int64_t B = x.size(0), H = x.size(1), W = x.size(2), C = x.size(3), Dm = w[kIn].size(0), hidden = w[kFc1].size(0), R = dt_proj.size(2);
    const int64_t bias_of[kLayers] = {Dm, C, hidden, C, C, C, Dm, Dm};
    for (size_t i = 0; i < kLayers; ++i)
        if (b[i].defined() && b[i].numel() != bias_of[i]) return py::none();              // (torch would broadcast one of another size)
    if (!has_shape(w[kIn], {Dm, C}) || !has_shape(w[kOut], {C, Dm}) || !has_shape(w[kFc1], {hidden, C}) || !has_shape(w[kFc2], {C, hidden}) ||
        w[kNorm].numel() != C || w[kNorm2].numel() != C || w[kOutNorm].numel() != Dm || !has_shape(w[kConv], {Dm, 1, 3, 3}) || R == 0 ||
        !has_shape(x_proj, {4, R + 2, Dm}) || !has_shape(dt_proj, {4, Dm, R}))
        return py::none();
    for (const at::Tensor *t : {&A, &D, &dt_bias})
        if (t->numel() != 4 * Dm || t->scalar_type() != at::ScalarType::Float || !on(*t, x) || !t->is_contiguous()) return py::none();

    at::Tensor out = at::empty_like(x);
    ss2d_block_params p = {};
    ss2d_forward_core_params &c = p.core;
    c.batch = (int)B; c.dim = (int)Dm; c.height = c.padded_height = (int)H; c.width = c.padded_width = (int)W; c.rank = (int)R;
    c.dtype = c.norm_dtype = code; c.normalise = c.out_channel_last = 1; c.eps = (float)eps[2];
    c.x_proj_weight = x_proj.data_ptr(); c.dt_proj_weight = dt_proj.data_ptr(); c.A = A.data_ptr(); c.D = D.data_ptr(); c.delta_bias = dt_bias.data_ptr();
    c.norm_weight = ptr_of(w[kOutNorm]); c.norm_bias = ptr_of(b[kOutNorm]);
    p.d_model = (int)C; p.hidden = (int)hidden; p.norm_eps = (float)eps[0]; p.norm2_eps = (float)eps[1];
    p.x = x.data_ptr(); p.residual = ptr_of(residual);
    if (!residual.defined()) { p.norm_weight = ptr_of(w[kNorm]); p.norm_bias = ptr_of(b[kNorm]); }
    p.in_proj_weight = ptr_of(w[kIn]); p.in_proj_bias = ptr_of(b[kIn]); p.conv_weight = ptr_of(w[kConv]); p.conv_bias = ptr_of(b[kConv]);
    p.out_proj_weight = ptr_of(w[kOut]); p.out_proj_bias = ptr_of(b[kOut]); p.norm2_weight = ptr_of(w[kNorm2]); p.norm2_bias = ptr_of(b[kNorm2]);
    if (whole) { p.fc1_weight = ptr_of(w[kFc1]); p.fc2_weight = ptr_of(w[kFc2]); }
    p.fc1_bias = ptr_of(b[kFc1]); p.fc2_bias = ptr_of(b[kFc2]); p.out = out.data_ptr();
    const int64_t need = ss2d_block_workspace_bytes(&p);
    if (need == SS2D_ENOTSUP) return py::none();
    if (need < 0) return py::int_(need);
    at::Tensor workspace = at::empty({need}, x.options().dtype(at::kByte));
    const int rc = enqueue(x, [&](void *stream) { return ss2d_block_fwd(&p, workspace.data_ptr(), need, stream); });
    if (rc == SS2D_ENOTSUP) return py::none();
    return rc != SS2D_OK ? py::object(py::int_(rc)) : py::cast(out);
}

// The scan's tensors, forward and backward: the caller's, as far as a kernel may have their addresses.
struct ScanTensors {
    at::Tensor u, delta, A, B, C, D, bias;
    int64_t batch, dim, L, N, groups, delta_dim;
    int code;

    // False for whatever csms6s.py refuses or has to look at itself.
    bool read(const py::tuple &kinds, const py::object &u_in, const py::object &delta_in, const py::object &A_in, const py::object &B_in,
              const py::object &C_in, const py::object &D_in, const py::object &bias_in) {
        bool ok = true;
        u = exactly(u_in, kinds, ok); delta = exactly(delta_in, kinds, ok); A = exactly(A_in, kinds, ok); B = exactly(B_in, kinds, ok);
        C = exactly(C_in, kinds, ok); D = exactly(D_in, kinds, ok); bias = exactly(bias_in, kinds, ok);
        if (!ok) return false;
        for (const at::Tensor *t : {&u, &delta, &A, &B, &C})
            if (!t->defined() || !plain(*t) || !on(*t, u) || t->numel() == 0) return false;
        code = dtype_code(u.scalar_type());
        if (code < 0 || u.dim() != 3 || delta.dim() != 3 || A.dim() != 2 || B.dim() != 4 || C.dim() != 4 || A.scalar_type() != at::kFloat) return false;
        batch = u.size(0); dim = u.size(1); L = u.size(2); N = A.size(1); groups = B.size(1); delta_dim = delta.size(1);
        for (const at::Tensor *t : {&u, &delta, &B, &C})
            if (t->scalar_type() != u.scalar_type() || !(t->stride(-1) == 1 || t->size(-1) == 1)) return false;
        if (dim % groups != 0 || dim % delta_dim != 0 || N > 256 || batch > INT32_MAX || dim > INT32_MAX || L > INT32_MAX) return false;
        if (!has_shape(delta, {batch, delta_dim, L}) || !has_shape(A, {dim, N}) || !has_shape(B, {batch, groups, N, L}) || !has_shape(C, {batch, groups, N, L}))
            return false;
        if (D.defined() && (D.scalar_type() != at::kFloat || !on(D, u) || !plain(D) || !has_shape(D, {dim}) || !D.is_contiguous())) return false;
        return !bias.defined() || (bias.scalar_type() == at::kFloat && on(bias, u) && plain(bias) && has_shape(bias, {delta_dim}) && bias.is_contiguous());
    }

    template <typename P> void describe(P &p, bool softplus) const {
        p.batch = (int)batch; p.dim = (int)dim; p.seqlen = (int)L; p.dstate = (int)N; p.n_groups = (int)groups; p.delta_dim = (int)delta_dim;
        p.in_dtype = code; p.delta_softplus = softplus ? 1 : 0;
        p.u = u.data_ptr(); p.delta = delta.data_ptr(); p.A = A.data_ptr(); p.B = B.data_ptr(); p.C = C.data_ptr();
        p.D = ptr_of(D); p.delta_bias = ptr_of(bias);
        p.u_batch_stride = u.stride(0); p.u_d_stride = u.stride(1);
        p.delta_batch_stride = delta.stride(0); p.delta_d_stride = delta.stride(1);
        p.A_d_stride = A.stride(0); p.A_dstate_stride = A.stride(1);
        p.B_batch_stride = B.stride(0); p.B_group_stride = B.stride(1); p.B_dstate_stride = B.stride(2);
        p.C_batch_stride = C.stride(0); p.C_group_stride = C.stride(1); p.C_dstate_stride = C.stride(2);
    }
};

// csms6s.py:selective_scan_fwd -- [out, x], None where its own checks have to speak, or the status of a failed call.
static py::object scan_fwd(const py::tuple &kinds, const py::object &u, const py::object &delta, const py::object &A, const py::object &B, const py::object &C,
                           const py::object &D, const py::object &bias, bool softplus, bool out_float, bool want_x) {
    ScanTensors t;
    if (!t.read(kinds, u, delta, A, B, C, D, bias)) return py::none();
    const auto f32 = t.u.options().dtype(at::kFloat);
    at::Tensor out = at::empty({t.batch, t.dim, t.L}, out_float ? f32 : t.u.options()), x;
    if (want_x) x = at::empty({t.batch, t.dim, (t.L + SS2D_SCAN_CHUNK - 1) / SS2D_SCAN_CHUNK, 2 * t.N}, f32);
    ss2d_scan_params p = {};
    t.describe(p, softplus);
    p.out_dtype = out_float ? SS2D_F32 : t.code;
    p.out = out.data_ptr(); p.x = want_x ? x.data_ptr() : nullptr;
    p.out_batch_stride = out.stride(0); p.out_d_stride = out.stride(1);
    const int rc = enqueue(t.u, [&](void *stream) { return ss2d_selective_scan_fwd(&p, stream); });
    if (rc != SS2D_OK) return py::int_(rc);
    py::list result(2);
    result[0] = py::cast(out);
    result[1] = want_x ? py::cast(x) : py::none();
    return result;
}

// csms6s.py:selective_scan_bwd, a delta row per channel -- the seven gradients (None for one that is not asked for), None or a status as above.
static py::object scan_bwd(const py::tuple &kinds, const py::object &u, const py::object &delta, const py::object &A, const py::object &B, const py::object &C,
                           const py::object &D, const py::object &bias, const py::object &dout_in, bool softplus) {
    ScanTensors t;
    bool ok = true;
    const at::Tensor dout = exactly(dout_in, kinds, ok);
    if (!ok || !dout.defined() || !t.read(kinds, u, delta, A, B, C, D, bias) || t.delta_dim != t.dim) return py::none();
    if (!plain(dout) || !on(dout, t.u) || !has_shape(dout, {t.batch, t.dim, t.L}) || !(dout.stride(-1) == 1 || t.L == 1) ||
        (dout.scalar_type() != t.u.scalar_type() && dout.scalar_type() != at::kFloat))
        return py::none();
    const auto f32 = t.u.options().dtype(at::kFloat);
    at::Tensor du = at::empty({t.batch, t.dim, t.L}, t.u.options()), ddelta = at::empty({t.batch, t.dim, t.L}, t.u.options());
    // sums, cleared in one launch
    at::Tensor sums[5] = {at::empty({t.dim, t.N}, f32), at::empty({t.batch, t.groups, t.N, t.L}, f32), at::empty({t.batch, t.groups, t.N, t.L}, f32)};
    if (t.D.defined()) sums[3] = at::empty({t.dim}, f32);
    if (t.bias.defined()) sums[4] = at::empty({t.dim}, f32);
    at::Tensor &dA = sums[0], dB = sums[1], dC = sums[2];
    void *ptrs[5];
    int64_t bytes[5];
    int n = 0;
    for (const at::Tensor &s : sums)
        if (s.defined()) { ptrs[n] = s.data_ptr(); bytes[n++] = 4 * s.numel(); }
    if (t.code != SS2D_F32) { dB = at::empty(sums[1].sizes(), t.u.options()); dC = at::empty(sums[2].sizes(), t.u.options()); }
    ss2d_scan_bwd_params p = {};
    t.describe(p, softplus);
    p.dout_dtype = dtype_code(dout.scalar_type());
    p.dout = dout.data_ptr(); p.dout_batch_stride = dout.stride(0); p.dout_d_stride = dout.stride(1);
    p.du = du.data_ptr(); p.ddelta = ddelta.data_ptr(); p.dA = dA.data_ptr(); p.dB = sums[1].data_ptr(); p.dC = sums[2].data_ptr();
    p.dD = sums[3].defined() ? sums[3].data_ptr() : nullptr;
    p.ddelta_bias = sums[4].defined() ? sums[4].data_ptr() : nullptr;
    const int rc = enqueue(t.u, [&](void *stream) {
        int status = ss2d_clear(ptrs, bytes, n, stream);
        if (status == SS2D_OK) status = ss2d_selective_scan_bwd(&p, stream);
        if (status == SS2D_OK && t.code != SS2D_F32)
            status = ss2d_round_pair((const float *)p.dB, dB.data_ptr(), dB.numel(), (const float *)p.dC, dC.data_ptr(), dC.numel(), t.code, stream);
        return status;
    });
    if (rc != SS2D_OK) return py::int_(rc);
    py::list result(7);
    const at::Tensor grads[7] = {du, ddelta, dA, dB, dC, sums[3], sums[4]};
    for (size_t i = 0; i < 7; ++i) result[i] = grads[i].defined() ? py::cast(grads[i]) : py::none();
    return result;
}

// csm.py:cross_scan_hip and cross_merge_hip (pairwise): the result, None or a status as above.
static py::object cross_scan(const py::tuple &kinds, const py::object &x_in) {
    bool ok = true;
    const at::Tensor x = exactly(x_in, kinds, ok);
    if (!ok || !x.defined() || x.dim() != 4 || x.numel() == 0 || !x.is_cuda() || !plain(x) || !x.is_contiguous()) return py::none();
    const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
    if (B > INT32_MAX || C > INT32_MAX || H > INT32_MAX || W > INT32_MAX) return py::none();
    at::Tensor y = at::empty({B, 4, C, H * W}, x.options());
    const int rc = enqueue(x, [&](void *stream) { return ss2d_cross_scan(x.data_ptr(), y.data_ptr(), (int)B, (int)C, (int)H, (int)W, (int)x.element_size(), stream); });
    return rc != SS2D_OK ? py::object(py::int_(rc)) : py::cast(y);
}

static py::object cross_merge(const py::tuple &kinds, const py::object &y_in) {
    bool ok = true;
    const at::Tensor y = exactly(y_in, kinds, ok);
    if (!ok || !y.defined() || y.dim() != 5 || y.numel() == 0 || y.size(1) != 4 || !y.is_cuda() || !plain(y) || !y.is_contiguous()) return py::none();
    const int64_t B = y.size(0), C = y.size(2), H = y.size(3), W = y.size(4);
    const int code = dtype_code(y.scalar_type());
    if (code < 0 || B > INT32_MAX || C > INT32_MAX || H > INT32_MAX || W > INT32_MAX) return py::none();
    at::Tensor out = at::empty({B, C, H * W}, y.options());
    const int rc = enqueue(y, [&](void *stream) {
        return ss2d_cross_merge(y.data_ptr(), out.data_ptr(), (int)B, (int)C, (int)H, (int)W, code, SS2D_MERGE_PAIRWISE, stream);
    });
    return rc != SS2D_OK ? py::object(py::int_(rc)) : py::cast(out);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("forward_core", &forward_core);
    m.def("block", &block);
    m.def("scan_fwd", &scan_fwd);
    m.def("scan_bwd", &scan_bwd);
    m.def("cross_scan", &cross_scan);
    m.def("cross_merge", &cross_merge);
}
