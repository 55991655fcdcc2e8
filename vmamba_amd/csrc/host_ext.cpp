// The host's share of forward_core and of a block of few positions, in C++: the checks of their tensors, the outputs and workspaces and
// the one call into the C ABI.  Through ctypes and torch's Python interface that took 14 us of a forward_core whose three kernels
// run for 18, and 20 us of a block; no kernel lives here, and what is checked is what the Python callers (core.py, block.py) checked.
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

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("forward_core", &forward_core);
    m.def("block", &block);
}
