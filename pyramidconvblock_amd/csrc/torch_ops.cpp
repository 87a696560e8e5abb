// The operators' host path in native code: allocation of results, argument checks, autograd nodes and the calls of
// libpdw.so for ConvBlock and OptimizedDepthwiseConv2d.  From Python, with torch.autograd.Function and ctypes, one
// training step of a block cost 250-900 us of host time (one interpreter-level call per launch, 10-20 us each, where the
// library's kernels run 3-30 us each); a Node here is entered by the autograd engine without the interpreter lock.
// Plain C++ (no device code): built with the host compiler against torch's headers and linked to libpdw.so beside it.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/pdw.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return PDW_F32;
        case at::kHalf: return PDW_F16;
        case at::kBFloat16: return PDW_BF16;
        default: return -1;
    }
}

void check(int status, const char* what) {
    TORCH_CHECK(status == 0, what, ": ", pdw_last_error(), " (status ", status, ")");
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Contiguous and 16-byte aligned (the kernels move 16-byte pieces; a view at an odd storage offset is copied).
Tensor dense(const Tensor& t) {
    Tensor c = t.is_contiguous() ? t : t.contiguous();
    return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone(at::MemoryFormat::Contiguous);
}

// What a node keeps of an input: the input itself where it went to the kernels as it is, so that a later change of it in
// place is noticed, else the copy that they read.
SavedVariable save(const Tensor& in, const Tensor& read) { return SavedVariable(read.is_same(in) ? in : read, false); }

// What a node has saved, as it comes back: a saved-tensor hook may have put another tensor in its place, and the kernels
// take addresses.  (Of another type: converted.)
Tensor restored(const SavedVariable& v, const std::shared_ptr<torch::autograd::Node>& node, at::IntArrayRef sizes,
                at::ScalarType type, c10::Device device) {
    Tensor t = v.unpack(node);
    TORCH_CHECK(t.defined() && t.sizes() == sizes && t.device() == device, node->name(),
                ": a saved tensor came back as another one (", sizes, " on ", device, " was saved)");
    return t.scalar_type() == type ? t : t.to(type);
}

// The gradient of a node's only output; zeros where the engine has none (a later node's backward returned none), as
// torch.autograd.Function gives them, so that inputs and parameters get gradients of zero and not none.
Tensor output_gradient(const torch::autograd::Node& node, const variable_list& grads) {
    return grads[0].defined() ? grads[0] : node.input_metadata(0).zeros_like();
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

Tensor bytes(size_t n, const Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// Whether a call belongs to the nodes below.  They have no forward-mode derivative and no batching rule, so such calls go
// on to the torch.autograd.Function forms, which refuse them; and a trace (torch.jit.trace) would record of them the
// allocation of the result alone, where a Function becomes a node of the graph that calls it again.
bool plain_call(const Tensor* in, int n) {
    if (torch::jit::tracer::isTracing()) return false;
    if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode)) return false;
    for (int i = 0; i < n; ++i)
        if (in[i].defined() && in[i]._fw_grad(0).defined()) return false;
    return true;
}

// ---------------------------------------------------------------------------------------------------------------
// The block

struct BlockShape {
    int B, H, W, h, w, D, I, K, dtype;
};

#define PDW_SHAPE(s) (s).B, (s).H, (s).W, (s).h, (s).w, (s).D, (s).I, (s).K, (s).dtype

enum { kX, kUp, kOut, kBOut, kPool, kBPool, kDw0, kDw1, kBlockInputs };   // order of a block's differentiable inputs

struct BlockNode : public torch::autograd::Node {
    SavedVariable x, w_up, w_out, w_pool, w_dw0, w_dw1, saved;
    BlockShape s;
    int64_t saved_bytes;
    bool has_b_out, has_b_pool;

    std::string name() const override { return "ConvBlockBackward"; }

    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* v : {&x, &w_up, &w_out, &w_pool, &w_dw0, &w_dw1, &saved}) v->reset_data();
    }

    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(kBlockInputs);
        const Tensor grad = output_gradient(*this, grads);
        // (unpacked first: a saved-tensor hook may run a whole recorded forward, as checkpointing does)
        const auto self = shared_from_this();
        const auto type = grad.scalar_type();   // (the engine has cast it to the output's type and checked its sizes)
        auto take = [&](const SavedVariable& v, std::initializer_list<int64_t> n) { return restored(v, self, n, type, grad.device()); };
        Tensor xs = take(x, {s.B, s.H, s.W, s.D}), wu = take(w_up, {s.I, s.D}), wo = take(w_out, {s.D, s.I}),
               wp = take(w_pool, {s.D, s.D}), d0 = take(w_dw0, {s.K, s.K, s.I}), d1 = take(w_dw1, {s.K, s.K, s.I});
        Tensor keep = restored(saved, self, {saved_bytes}, at::kByte, grad.device());
        at::AutoDispatchBelowADInplaceOrView below;
        for (Tensor* t : {&xs, &wu, &wo, &wp, &d0, &d1, &keep}) *t = dense(*t);
        const Tensor gy = dense(grad);
        const c10::DeviceGuard guard(xs.device());
        auto like = [](const Tensor& t) { return at::empty(t.sizes(), t.options()); };
        if (task_should_compute_output(kX)) out[kX] = like(xs);
        out[kUp] = like(wu), out[kOut] = like(wo), out[kPool] = like(wp), out[kDw0] = like(d0), out[kDw1] = like(d1);
        if (has_b_out) out[kBOut] = at::empty({s.D}, xs.options());
        if (has_b_pool) out[kBPool] = at::empty({s.D}, xs.options());
        const Tensor ws = bytes(pdw_block_bwd_workspace_bytes(PDW_SHAPE(s)), xs);
        check(pdw_block_bwd(ptr(gy), ptr(xs), ptr(keep), ptr(wu), ptr(d0), ptr(d1), ptr(wp), ptr(wo), ptr(out[kX]),
                            ptr(out[kUp]), ptr(out[kDw0]), ptr(out[kDw1]), ptr(out[kPool]), ptr(out[kBPool]),
                            ptr(out[kOut]), ptr(out[kBOut]), ptr(ws), ws.numel(), PDW_SHAPE(s), stream_of(xs)),
              "pdw_block_bwd");
        return out;
    }
};

// Whether these are a block of the library's calls: everything on x's device in x's type, conv_up without bias, two square
// filters of one shape, widths that fit together.  (Which extents, widths and filters are covered, the library says.)
bool block_args(const Tensor* in, const Tensor& b_up, double s0, double s1, BlockShape* s) {
    const Tensor& x = in[kX];
    if (b_up.defined() || s0 != 1.0 || s1 == 1.0 || x.dim() != 4 || !x.is_cuda()) return false;
    const int dt = dtype_code(x.scalar_type());
    if (dt < 0) return false;
    for (int i = 1; i < kBlockInputs; ++i)
        if (in[i].defined() && (in[i].scalar_type() != x.scalar_type() || in[i].device() != x.device())) return false;
    const Tensor &up = in[kUp], &out = in[kOut], &pool = in[kPool], &d0 = in[kDw0], &d1 = in[kDw1];
    if (up.dim() != 2 || out.dim() != 2 || pool.dim() != 2 || d0.dim() != 3 || d0.sizes() != d1.sizes()) return false;
    const int64_t D = x.size(3), I = up.size(0), K = d0.size(0);
    if (up.size(1) != D || d0.size(1) != K || d0.size(2) != I || out.size(0) != D || out.size(1) != I || (I & 1) ||
        pool.size(0) != D || pool.size(1) != D)
        return false;
    for (int i : {kBOut, kBPool})
        if (in[i].defined() && (in[i].dim() != 1 || in[i].size(0) != D)) return false;
    for (int64_t e : x.sizes())
        if (e > 0x7fffffff) return false;
    const int H = (int)x.size(1), W = (int)x.size(2);
    *s = {(int)x.size(0), H, W, (int)(H * s1), (int)(W * s1), (int)D, (int)I, (int)K, dt};
    return true;
}

// Whether the inference call of the fused launches takes it.
bool infer_shape(const BlockShape& s) {
    return s.H == 2 * s.h && s.W == 2 * s.w && pdw_convblock_supported(s.B, s.H, s.W, s.D, s.I, s.K, s.dtype);
}

Tensor block_train_or_infer(const Tensor* in, const BlockShape& s, bool grad) {
    const c10::DeviceGuard guard(in[kX].device());
    Tensor d[kBlockInputs], y, saved;
    std::shared_ptr<BlockNode> node;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        for (int i = 0; i < kBlockInputs; ++i)
            if (in[i].defined()) d[i] = dense(in[i]);
        y = at::empty(d[kX].sizes(), d[kX].options());
        saved = bytes(pdw_block_saved_bytes(PDW_SHAPE(s)), d[kX]);
        check(pdw_block_fwd(ptr(d[kX]), ptr(d[kUp]), ptr(d[kDw0]), ptr(d[kDw1]), ptr(d[kPool]), ptr(d[kBPool]),
                            ptr(d[kOut]), ptr(d[kBOut]), ptr(y), ptr(saved), saved.numel(), PDW_SHAPE(s), stream_of(y)),
              "pdw_block_fwd");
    }
    if (grad) {
        node = std::shared_ptr<BlockNode>(new BlockNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(in[kX], in[kUp], in[kOut], in[kBOut], in[kPool],
                                                                 in[kBPool], in[kDw0], in[kDw1]));
        auto keep = [&](int i) { return save(in[i], d[i]); };
        node->x = keep(kX), node->w_up = keep(kUp), node->w_out = keep(kOut), node->w_pool = keep(kPool);
        node->w_dw0 = keep(kDw0), node->w_dw1 = keep(kDw1), node->saved = SavedVariable(saved, false);
        node->s = s, node->saved_bytes = saved.numel(), node->has_b_out = in[kBOut].defined(), node->has_b_pool = in[kBPool].defined();
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------------------------
// The depthwise convolution

struct ConvGeo {
    int sh, sw, ph, pw, dh, dw;
};

#define PDW_CONV(x, w, g)                                                                                         \
    (int)(x)[0], (int)(x)[1], (int)(x)[2], (int)(x)[3], (int)(w)[0], (int)(w)[1], (g).sh, (g).sw, (g).ph, (g).pw, \
        (g).dh, (g).dw

struct ConvNode : public torch::autograd::Node {
    SavedVariable x, w;
    at::DimVector x_sizes, w_sizes;
    ConvGeo g;
    at::ScalarType x_type;

    std::string name() const override { return "DepthwiseConv2DBackward"; }

    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x.reset_data(), w.reset_data();
    }

    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(2);
        const Tensor grad = output_gradient(*this, grads);
        const auto self = shared_from_this();   // (unpacked first, as in BlockNode)
        const Tensor w_saved = restored(w, self, w_sizes, grad.scalar_type(), grad.device()),
                     x_saved = restored(x, self, x_sizes, grad.scalar_type(), grad.device());
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor wd = dense(w_saved), xd = dense(x_saved), gy = dense(grad);
        const c10::DeviceGuard guard(xd.device());
        const int dt = dtype_code(wd.scalar_type());
        void* const stream = stream_of(xd);
        const auto xs = xd.sizes(), ws = wd.sizes();
        const bool empty = xd.numel() == 0 || gy.numel() == 0;
        const bool want_x = task_should_compute_output(0), want_w = task_should_compute_output(1);
        Tensor dx, dw, work;
        if (want_x) dx = at::empty(xs, xd.options());
        if (want_w) dw = at::empty(ws, wd.options());
        if (want_w && !empty) work = bytes(pdw_dwconv_wgrad_workspace_bytes(PDW_CONV(xs, ws, g), dt) + 4, xd);
        if (empty) {
            if (want_x) dx.zero_();
            if (want_w) dw.zero_();
        } else if (want_x && want_w) {
            check(pdw_dwconv_bwd(ptr(gy), ptr(wd), ptr(xd), ptr(dx), ptr(dw), ptr(work), work.numel(), PDW_CONV(xs, ws, g), dt, stream),
                  "pdw_dwconv_bwd");
        } else if (want_x) {
            check(pdw_dwconv_dgrad(ptr(gy), ptr(wd), ptr(dx), PDW_CONV(xs, ws, g), dt, stream), "pdw_dwconv_dgrad");
        } else if (want_w) {
            check(pdw_dwconv_wgrad(ptr(xd), ptr(gy), ptr(dw), ptr(work), work.numel(), PDW_CONV(xs, ws, g), dt, stream), "pdw_dwconv_wgrad");
        }
        if (want_x) out[0] = dx.to(x_type);
        if (want_w) out[1] = dw;
        return out;
    }
};

Tensor conv_forward(const Tensor& x, const Tensor& w, const ConvGeo& g) {
    TORCH_CHECK_VALUE(x.dim() == 4 && w.dim() == 3 && x.size(3) == w.size(2),
                      "expected input [B,H,W,C] and weight [k1,k2,C], got ", x.sizes(), " and ", w.sizes());
    TORCH_CHECK(x.is_cuda() && w.is_cuda(), "pyramid dwconv kernels run on a HIP device only (tensor is on ",
                (x.is_cuda() ? w : x).device(), "); there is no CPU path");
    TORCH_CHECK(x.device() == w.device(), "tensors on different devices: ", x.device(), " vs ", w.device());
    TORCH_CHECK_TYPE(dtype_code(w.scalar_type()) >= 0, "pyramid dwconv kernels support float32/float16/bfloat16, got ",
                     w.scalar_type());
    const c10::DeviceGuard guard(x.device());
    const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad());
    Tensor y, xd, wd;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        xd = dense(x.scalar_type() == w.scalar_type() ? x : x.to(w.scalar_type())), wd = dense(w);
        const auto xs = xd.sizes(), ws = wd.sizes();
        const int oh = pdw_conv_out_size((int)xs[1], (int)ws[0], g.sh, g.ph, g.dh);
        const int ow = pdw_conv_out_size((int)xs[2], (int)ws[1], g.sw, g.pw, g.dw);
        y = at::empty({xs[0], oh, ow, xs[3]}, xd.options());
        if (y.numel())
            check(pdw_dwconv_fwd(ptr(xd), ptr(wd), ptr(y), PDW_CONV(xs, ws, g), dtype_code(wd.scalar_type()), stream_of(xd)),
                  "pdw_dwconv_fwd");
    }
    if (grad) {
        auto node = std::shared_ptr<ConvNode>(new ConvNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, w));
        // (what the kernels read, as in block_train_or_infer: a copy is not made again by the backward, and stays valid
        // when its source is changed in place)
        node->x = save(x, xd), node->w = save(w, wd);
        node->x_sizes = x.sizes(), node->w_sizes = w.sizes();
        node->g = g, node->x_type = x.scalar_type();
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------------------------
// Python entry points

bool tensor_arg(PyObject* o, Tensor* t) {
    if (o == Py_None) return true;
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a Tensor or None, got %s", Py_TYPE(o)->tp_name);
        return false;
    }
    *t = THPVariable_Unpack(o);
    return true;
}

// block(x, w_up, b_up, w_out, b_out, w_pool, b_pool, w_dw0, w_dw1, s0, s1): the block's output; None where ConvBlockFunction
// has to answer (a case that the library's block calls do not cover, a transform, a trace); True where no gradient is wanted and its inference call (block_infer) covers it.
PyObject* py_block(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 11, "block: 11 arguments expected");
    Tensor in[kBlockInputs], b_up;
    Tensor* const slot[9] = {&in[kX], &in[kUp], &b_up, &in[kOut], &in[kBOut], &in[kPool], &in[kBPool], &in[kDw0], &in[kDw1]};
    for (int i = 0; i < 9; ++i)
        if (!tensor_arg(args[i], slot[i])) return nullptr;
    const double s0 = PyFloat_AsDouble(args[9]), s1 = PyFloat_AsDouble(args[10]);
    if (PyErr_Occurred()) return nullptr;
    BlockShape s;
    if (!plain_call(in, kBlockInputs) || !block_args(in, b_up, s0, s1, &s)) Py_RETURN_NONE;
    bool grad = false;
    if (at::GradMode::is_enabled())
        for (const Tensor& t : in) grad = grad || (t.defined() && t.requires_grad());
    if (!grad && infer_shape(s)) Py_RETURN_TRUE;
    if (!pdw_block_supported(PDW_SHAPE(s))) Py_RETURN_NONE;
    Tensor y;
    {
        pybind11::gil_scoped_release no_gil;
        y = block_train_or_infer(in, s, grad);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// block_infer(x, w_up, w_out, b_out, w_pool, b_pool, w_dw0, w_dw1): pdw_convblock_infer, refused where block() would not
// name it.
PyObject* py_block_infer(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == kBlockInputs, "block_infer: 8 arguments expected");
    Tensor in[kBlockInputs];
    for (int i = 0; i < kBlockInputs; ++i) {
        if (!tensor_arg(args[i], &in[i])) return nullptr;
    }
    // (the kernels take addresses: a tensor of another device, type or size must not get that far)
    for (int i = 0; i < kBlockInputs; ++i)
        TORCH_CHECK(in[i].defined() ? in[i].is_cuda() : i == kBOut || i == kBPool,
                    "convblock_infer: tensors on a HIP device expected (the biases may be None)");
    BlockShape s;
    TORCH_CHECK(plain_call(in, kBlockInputs) && block_args(in, Tensor(), 1.0, 0.5, &s) && infer_shape(s),
                "convblock_infer: not a call that pdw_convblock_infer covers (input ", in[kX].sizes(), " ",
                in[kX].scalar_type(), ", filters ", in[kDw0].sizes(), ")");
    Tensor y;
    {
        pybind11::gil_scoped_release no_gil;
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(in[kX].device());
        for (Tensor& t : in)
            if (t.defined()) t = dense(t);
        const Tensor& x = in[kX];
        y = at::empty(x.sizes(), x.options());
        const Tensor ws = bytes(pdw_convblock_infer_workspace_bytes(s.B, s.H, s.W, s.D, s.I, s.K, s.dtype), x);
        check(pdw_convblock_infer(ptr(x), ptr(in[kUp]), ptr(in[kDw0]), ptr(in[kDw1]), ptr(in[kPool]), ptr(in[kBPool]),
                                  ptr(in[kOut]), ptr(in[kBOut]), ptr(y), ptr(ws), ws.numel(), s.B, s.H, s.W, s.D, s.I, s.K, s.dtype, stream_of(x)),
              "pdw_convblock_infer");
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// dwconv(x, w, (sh, sw), (ph, pw), (dh, dw)): the convolution's output; None where DepthwiseConv2DFunction has to answer.
PyObject* py_dwconv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 5, "dwconv: 5 arguments expected");
    Tensor in[2];
    if (!tensor_arg(args[0], &in[0]) || !tensor_arg(args[1], &in[1])) return nullptr;
    const Tensor &x = in[0], &w = in[1];
    if (!plain_call(in, 2)) Py_RETURN_NONE;
    int v[6];
    for (int i = 0; i < 3; ++i)
        if (!PyArg_ParseTuple(args[2 + i], "ii", &v[2 * i], &v[2 * i + 1])) return nullptr;
    Tensor y;
    {
        pybind11::gil_scoped_release no_gil;
        y = conv_forward(x, w, {v[0], v[1], v[2], v[3], v[4], v[5]});
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"block", (PyCFunction)(void (*)(void))py_block, METH_FASTCALL, nullptr},
    {"block_infer", (PyCFunction)(void (*)(void))py_block_infer, METH_FASTCALL, nullptr},
    {"dwconv", (PyCFunction)(void (*)(void))py_dwconv, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_pdw_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pdw_torch(void) { return PyModule_Create(&kModule); }
