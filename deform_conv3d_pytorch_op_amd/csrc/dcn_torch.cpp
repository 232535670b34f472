// The autograd layer of the package in C++: `_native.conv_offset` and `_native.conv2d` check a call, run
// the operators of libdcn_amd.so on the current stream and record the backward node; the `_forward` and
// `_backward` entries are their halves without a node, for the package's Python Functions.  In Python these
// steps cost more than the kernels of a small layer: every operator call converted some thirty arguments,
// and the backward half ran on the autograd engine's own thread, which had to take turns for the
// interpreter lock with the thread that waits for it (2 images of 16 x 16, 8 -> 8 channels, forward and
// backward: 190 us, of which the GPU worked 60).
//
// Replaces the host code of the reference's Functions
// (deform3d/deform_conv3d_functions/deform_conv3d_function.py:7-77,
// deform2d_double/deform_conv2d_functions/deform_conv2d_function.py:7-77, conv2d/conv2d_functions/conv2d_function.py:7-67)
// and, for the checks and their messages, of its shape_check (deform3d/lib/deform_conv3d_cuda.cpp:24-87).
#include "../../include/dcn_amd.h"

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

PyObject* g_library_error = nullptr;     // the package's exception for calls that the library rejects

void check(bool cond, const char* msg) {
    if (!cond) throw std::runtime_error(msg);
}
void check_rc(int rc) {
    if (rc == DCN_OK) return;
    const std::string msg = dcn_last_error();
    pybind11::gil_scoped_acquire gil;
    PyErr_SetString(g_library_error ? g_library_error : PyExc_RuntimeError, msg.c_str());
    throw pybind11::error_already_set();
}

struct Config {
    int nd = 0;
    int stride[3], pad[3], dil[3];
    int cpg = 0, group = 0;              // cpg = 0: the plain convolution
    bool standard = false, oob_zero = false;
};

// The library's geometry arguments, in the order of DCN3D_GEOMETRY / DCN2D_GEOMETRY / CONV2D_GEOMETRY.
struct Geometry {
    int v[23];
    size_t ws_bytes;
};

int dtype_index(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return 0;
        case at::kDouble: return 1;
        case at::kBFloat16: return 2;
        case at::kHalf: return 3;
        default: return -1;
    }
}

void device_check(const Tensor& t0, std::initializer_list<const Tensor*> others) {
    check(t0.is_cuda(), "deformable convolution runs on the GPU only: tensors must be on a HIP device "
                        "(there is no CPU path in this package)");
    check(dtype_index(t0.scalar_type()) >= 0, "dtype must be float32, float64, bfloat16 or float16");
    for (const Tensor* t : others) {
        if (!t->defined()) continue;
        check(t->device() == t0.device(), "all tensors must be on the same GPU");
        check(t->scalar_type() == t0.scalar_type(), "all tensors must have the same dtype");
    }
}

int64_t floor_div(int64_t a, int64_t b) { return a / b - ((a % b != 0) && ((a < 0) != (b < 0))); }

// Output extents: the reference's dilation-blind formula (deform3d/lib/deform_conv3d_cuda.cpp:15-17) or
// the usual dilation-aware one.
void output_size(const Config& c, const Tensor& input, const Tensor& weight, bool standard, int64_t* out) {
    for (int a = 0; a < c.nd; ++a) {
        check(c.stride[a] != 0, "stride must not be zero");
        const int64_t k = weight.size(2 + a), span = standard ? (int64_t)c.dil[a] * (k - 1) + 1 : k;
        out[a] = floor_div(input.size(2 + a) + 2 * (int64_t)c.pad[a] - span, c.stride[a]) + 1;
    }
}

Geometry geometry(const Config& c, const Tensor& input, const Tensor& weight, const int64_t* out) {
    Geometry g;
    int* v = g.v;
    *v++ = (int)input.size(0);
    *v++ = (int)input.size(1);
    *v++ = (int)weight.size(0);
    size_t in_v = 1, out_v = 1;
    int kv = 1;
    for (int a = 0; a < c.nd; ++a) { *v++ = (int)input.size(2 + a); in_v *= input.size(2 + a); }
    for (int a = 0; a < c.nd; ++a) { *v++ = (int)out[a]; out_v *= out[a]; }
    for (int a = 0; a < c.nd; ++a) { *v++ = (int)weight.size(2 + a); kv *= (int)weight.size(2 + a); }
    for (int a = 0; a < c.nd; ++a) *v++ = c.pad[a];
    for (int a = 0; a < c.nd; ++a) *v++ = c.stride[a];
    for (int a = 0; a < c.nd; ++a) *v++ = c.dil[a];
    const int elem = (int)input.element_size(), n = (int)input.size(0), ci = (int)input.size(1), co = (int)weight.size(0);
    if (c.cpg > 0) {
        *v++ = c.cpg;
        g.ws_bytes = dcn_workspace_bytes_for(elem, n, ci, co, in_v, out_v, kv, c.group, c.cpg);
    } else
        g.ws_bytes = conv2d_workspace_bytes(elem, n, ci, co, in_v, out_v, kv, c.group);
    *v++ = c.group;
    return g;
}

// The checks of the reference's shape_check with its messages; `shape`: of grad_output, in the backward pass.
void shape_check(const Config& c, const Tensor& input, const Tensor& weight, const Tensor& offset, int64_t* out, const at::IntArrayRef* shape = nullptr) {
    static const char* const out_msg[2][3] = {{"error outhh", "error outww", ""}, {"error output ll", "error outhh", "error outww"}};
    static const char* const off_msg[2][3] = {{"off h", "off w", ""}, {"off l", "off h", "off w"}};
    const int nd = c.nd;
    check(input.dim() == nd + 2, "input dim");
    check(weight.dim() == nd + 2, "kernel dim");
    output_size(c, input, weight, c.standard, out);
    check(input.size(1) == weight.size(1) * c.group, "input c != kernel c");
    if (shape) {
        check((int)shape->size() == nd + 2, "output dim");
        check((*shape)[0] == input.size(0), "output b != input b");
        check((*shape)[1] == weight.size(0), "ou c != ker c");
    }
    check(offset.dim() == nd + 2, "off dim");
    check(offset.size(0) == input.size(0), "off batch");
    int64_t kv = 1;
    for (int a = 0; a < nd; ++a) kv *= weight.size(2 + a);
    check(c.cpg > 0 && input.size(1) % c.cpg == 0, "off channel");
    check(offset.size(1) == input.size(1) / c.cpg * nd * kv, "off channel");
    for (int a = 0; a < nd; ++a) check(offset.size(2 + a) == (shape ? (*shape)[2 + a] : out[a]), off_msg[nd - 2][a]);
    for (int a = 0; a < nd; ++a)
        check(input.size(2 + a) + 2 * c.pad[a] - weight.size(2 + a) >= 0 && out[a] >= 1 && (!shape || (*shape)[2 + a] == out[a]), out_msg[nd - 2][a]);
    check(c.group > 0 && weight.size(0) % c.group == 0, "ou c != ker c");
}
void conv_check(const Config& c, const Tensor& input, const Tensor& weight, const Tensor& bias, int64_t* out) {
    check(weight.dim() == 4, "kernel dim");
    check(input.dim() == 4, "input dim");
    check(c.group > 0 && input.size(1) == weight.size(1) * c.group, "input c != kernel c");
    check(weight.size(0) % c.group == 0, "ou c != ker c");
    check(input.scalar_type() == at::kFloat || input.scalar_type() == at::kDouble, "dtype must be float32 or float64");
    device_check(input, {&weight, &bias});
    output_size(c, input, weight, true, out);
    check(out[0] >= 1, "error outhh");
    check(out[1] >= 1, "error outww");
}

// Calls an operator: its pointers, the geometry by value, then workspace and stream.
#define GEO3(g) g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12], g[13], g[14], g[15], g[16], g[17], g[18], \
                g[19], g[20], g[21], g[22]
#define GEO2(g) g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12], g[13], g[14], g[15], g[16]
#define GEOC(g) g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12], g[13], g[14], g[15]

struct Workspace {
    void* p;
    size_t n;
    void* stream;
};
template <typename T> const T* cptr(const Tensor& t) { return t.defined() ? static_cast<const T*>(t.const_data_ptr()) : nullptr; }
template <typename T> T* mptr(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }

int run_forward(int nd, int dt, const Tensor& in, const Tensor& w, const Tensor& off, const Tensor& bias, const Tensor& out, const int* g, const Workspace& ws) {
#define CALL(SUF, T)                                                                                                                                       \
    (nd == 3 ? dcn3d_forward_##SUF(cptr<T>(in), cptr<T>(w), cptr<T>(off), cptr<T>(bias), mptr<T>(out), GEO3(g), ws.p, ws.n, ws.stream)     \
             : dcn2d_forward_##SUF(cptr<T>(in), cptr<T>(w), cptr<T>(off), cptr<T>(bias), mptr<T>(out), GEO2(g), ws.p, ws.n, ws.stream))
    switch (dt) {
        case 0: return CALL(f32, float);
        case 1: return CALL(f64, double);
        case 2: return CALL(bf16, void);
        default: return CALL(f16, void);
    }
#undef CALL
}
int run_backward_data(int nd, int dt, bool oob_zero, const Tensor& in, const Tensor& w, const Tensor& off, const Tensor& go, const Tensor& gi, const Tensor& goff,
                      const int* g, const Workspace& ws) {
    if (nd == 3 && oob_zero) {          // the reference's 2-D kernels have no out-of-range term
        check(dt < 2, "oob_offset_grad='zero' is available in float32 and float64 only");
        if (dt == 0)
            return dcn3d_backward_input_offset_flags_f32(cptr<float>(in), cptr<float>(w), cptr<float>(off), cptr<float>(go), mptr<float>(gi), mptr<float>(goff),
                                                         GEO3(g), ws.p, ws.n, ws.stream, DCN_FLAG_OOB_OFFSET_GRAD_ZERO);
        return dcn3d_backward_input_offset_flags_f64(cptr<double>(in), cptr<double>(w), cptr<double>(off), cptr<double>(go), mptr<double>(gi), mptr<double>(goff),
                                                     GEO3(g), ws.p, ws.n, ws.stream, DCN_FLAG_OOB_OFFSET_GRAD_ZERO);
    }
#define CALL(SUF, T)                                                                                                                                     \
    (nd == 3 ? dcn3d_backward_input_offset_##SUF(cptr<T>(in), cptr<T>(w), cptr<T>(off), cptr<T>(go), mptr<T>(gi), mptr<T>(goff), GEO3(g), ws.p, ws.n, ws.stream) \
             : dcn2d_backward_input_offset_##SUF(cptr<T>(in), cptr<T>(w), cptr<T>(off), cptr<T>(go), mptr<T>(gi), mptr<T>(goff), GEO2(g), ws.p, ws.n, ws.stream))
    switch (dt) {
        case 0: return CALL(f32, float);
        case 1: return CALL(f64, double);
        case 2: return CALL(bf16, void);
        default: return CALL(f16, void);
    }
#undef CALL
}
int run_backward_weight(int nd, int dt, const Tensor& in, const Tensor& off, const Tensor& go, const Tensor& gw, const int* g, const Workspace& ws) {
#define CALL(SUF, T)                                                                                                                    \
    (nd == 3 ? dcn3d_backward_weight_##SUF(cptr<T>(in), cptr<T>(off), cptr<T>(go), mptr<T>(gw), GEO3(g), ws.p, ws.n, ws.stream) \
             : dcn2d_backward_weight_##SUF(cptr<T>(in), cptr<T>(off), cptr<T>(go), mptr<T>(gw), GEO2(g), ws.p, ws.n, ws.stream))
    switch (dt) {
        case 0: return CALL(f32, float);
        case 1: return CALL(f64, double);
        case 2: return CALL(bf16, void);
        default: return CALL(f16, void);
    }
#undef CALL
}

Tensor workspace_tensor(const Tensor& like, size_t bytes) {
    return at::empty({(int64_t)(bytes ? bytes : 1)}, like.options().dtype(at::kByte));
}
Workspace workspace(const Tensor& t, size_t bytes, hipStream_t stream) { return Workspace{t.data_ptr(), bytes, stream}; }

// DCN_OVERLAP_BACKWARD=1: backward_weight next to backward_input_offset on a second stream.  Off by
// default: a workgroup of the fused backward kernel takes nearly all of a CU's LDS, so the two kernels never
// share a CU; they only take turns, which upsets the order in which the fused kernel works through its
// items and measured slower than one stream (4.02 against 3.69 ms per step at 64 -> 64 channels, 16x56x56).
bool overlap_backward() {
    static const bool v = [] { const char* e = getenv("DCN_OVERLAP_BACKWARD"); return e && !strcmp(e, "1"); }();
    return v;
}
c10::hip::HIPStream side_stream(c10::DeviceIndex d) {         // one per device, default priority
    static std::mutex lock;
    static std::vector<c10::optional<c10::hip::HIPStream>> streams(64);
    std::lock_guard<std::mutex> guard(lock);
    auto& s = streams.at(d);
    if (!s) s = c10::hip::getStreamFromPool(false, d);
    return *s;
}
void wait_for(hipStream_t waiter, hipStream_t other) {
    hipEvent_t e;
    check(hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess && hipEventRecord(e, other) == hipSuccess &&
              hipStreamWaitEvent(waiter, e, 0) == hipSuccess && hipEventDestroy(e) == hipSuccess,
          "cannot order the two backward streams");
}

struct Gradients {
    Tensor input, offset, weight, bias;
};

Gradients conv_offset_backward(const Config& c, const Tensor& input, const Tensor& offset, const Tensor& weight, const Tensor& grad_output, bool need_data,
                               bool need_weight, bool need_bias) {
    device_check(input, {&offset, &weight, &grad_output});
    int64_t out[3];
    const at::IntArrayRef shape = grad_output.sizes();
    shape_check(c, input, weight, offset, out, &shape);
    const Geometry g = geometry(c, input, weight, out);
    const Tensor in = input.contiguous(), off = offset.contiguous(), w = weight.contiguous(), go = grad_output.contiguous();
    const int dt = dtype_index(in.scalar_type());
    check(!(c.nd == 3 && c.oob_zero && need_data && dt >= 2), "oob_offset_grad='zero' is available in float32 and float64 only");
    const hipStream_t main = c10::hip::getCurrentHIPStream(in.device().index()).stream();
    Gradients r;
    const bool two = need_data && need_weight && overlap_backward();
    if (need_weight) r.weight = two ? at::zeros_like(w) : at::empty_like(w);
    if (need_data) {
        r.input = two ? at::zeros_like(in) : at::empty_like(in);
        r.offset = at::empty_like(off);
    }
    if (two) {
        const Tensor ws = workspace_tensor(in, g.ws_bytes), ws_w = workspace_tensor(in, g.ws_bytes);
        const hipStream_t side = side_stream(in.device().index()).stream();
        wait_for(side, main);                            // the operands and the zero fills above are ready
        check_rc(run_backward_data(c.nd, dt, c.oob_zero, in, w, off, go, r.input, r.offset, g.v, workspace(ws, g.ws_bytes, main)));
        check_rc(run_backward_weight(c.nd, dt, in, off, go, r.weight, g.v, workspace(ws_w, g.ws_bytes, side)));
        wait_for(main, side);                            // everything issued later on the caller's stream sees grad_weight
    } else if (need_data || need_weight) {
        size_t in_v = 1, out_v = 1;
        int kv = 1;
        for (int a = 0; a < c.nd; ++a) { in_v *= in.size(2 + a); out_v *= out[a]; kv *= (int)w.size(2 + a); }
        const size_t bytes = dcn_layer_backward_workspace_bytes((int)in.element_size(), c.nd, g.v[0], g.v[1], g.v[2], in_v, out_v, kv, c.group, c.cpg);
        const Tensor ws = workspace_tensor(in, bytes);
        const bool bias_too = need_bias && need_weight;
        if (bias_too) r.bias = at::empty({w.size(0)}, w.options());
        auto p = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
        check_rc(dcn_layer_backward(c.nd, dt, cptr<void>(in), cptr<void>(w), cptr<void>(off), cptr<void>(go), p(r.input), p(r.offset), p(r.weight), p(r.bias), g.v,
                                    ws.data_ptr(), bytes, main, c.nd == 3 && c.oob_zero ? DCN_FLAG_OOB_OFFSET_GRAD_ZERO : 0u));
        if (bias_too) return r;
    }
    if (need_bias) {
        static const int64_t dims[2][4] = {{0, 2, 3, 0}, {0, 2, 3, 4}};
        r.bias = go.sum(at::IntArrayRef(dims[c.nd - 2], c.nd + 1));
    }
    return r;
}

Gradients conv2d_backward(const Config& c, const Tensor& input, const Tensor& weight, const Tensor& grad_output, bool need_data, bool need_weight, bool need_bias) {
    int64_t out[3];
    conv_check(c, input, weight, grad_output, out);
    check(grad_output.dim() == 4, "output dim");
    check(grad_output.size(0) == input.size(0), "output b != input b");
    check(grad_output.size(1) == weight.size(0), "ou c != ker c");
    check(grad_output.size(2) == out[0], "error outhh");
    check(grad_output.size(3) == out[1], "error outww");
    const Geometry geo = geometry(c, input, weight, out);
    const int* g = geo.v;
    const Tensor in = input.contiguous(), w = weight.contiguous(), go = grad_output.contiguous();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(in.device().index()).stream();
    const size_t bytes = conv2d_layer_backward_workspace_bytes((int)in.element_size(), g[0], g[1], g[2], (size_t)(in.size(2) * in.size(3)), (size_t)(out[0] * out[1]),
                                                               (int)(w.size(2) * w.size(3)), c.group);
    check(bytes > 0, "inconsistent convolution geometry");
    Gradients r;
    if (need_data) r.input = at::empty_like(in);
    if (need_weight) r.weight = at::empty_like(w);
    if (need_weight && need_bias) r.bias = at::empty({w.size(0)}, w.options());
    if (need_data || need_weight) {
        const Tensor ws = workspace_tensor(in, bytes);
        auto p = [](const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
#define CALL(SUF, T) conv2d_layer_backward_##SUF(cptr<T>(in), cptr<T>(w), cptr<T>(go), (T*)p(r.input), (T*)p(r.weight), (T*)p(r.bias), GEOC(g), ws.data_ptr(), bytes, stream)
        check_rc(in.scalar_type() == at::kFloat ? CALL(f32, float) : CALL(f64, double));
#undef CALL
    }
    if (need_bias && !need_weight) r.bias = go.sum(at::IntArrayRef({0, 2, 3}));
    return r;
}

// The backward node of either layer: edges input, offset (deformable layers), weight, bias (if given).
struct LayerBackward : public Node {
    Config cfg;
    SavedVariable input_, offset_, weight_;
    bool has_bias = false;

    std::string name() const override { return cfg.cpg == 0 ? "Conv2dFunctionBackward" : cfg.nd == 3 ? "ConvOffset3dFunctionBackward" : "ConvOffset2dFunctionBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        input_.reset_data();
        offset_.reset_data();
        weight_.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const bool deform = cfg.cpg > 0;
        const size_t at_w = deform ? 2 : 1, n = at_w + 1 + (has_bias ? 1 : 0);
        variable_list res(n);
        // (a gradient that is not defined is zeros, as for a Function)
        const Tensor grad_output = grads[0].defined() ? grads[0] : input_metadata(0).zeros_like();
        const Tensor input = input_.unpack(), weight = weight_.unpack(), offset = deform ? offset_.unpack() : Tensor();
        const bool need_in = task_should_compute_output(0), need_off = deform && task_should_compute_output(1);
        const bool need_w = task_should_compute_output(at_w), need_b = has_bias && task_should_compute_output(at_w + 1);
        const bool create_graph = c10::GradMode::is_enabled();
        {
            c10::AutoGradMode off_mode(false);
            const c10::OptionalDeviceGuard guard(input.device());
            Gradients g = deform ? conv_offset_backward(cfg, input, offset, weight, grad_output, need_in || need_off, need_w, need_b)
                                 : conv2d_backward(cfg, input, weight, grad_output, need_in, need_w, need_b);
            if (need_in) res[0] = std::move(g.input);
            if (need_off) res[1] = std::move(g.offset);
            if (need_w) res[at_w] = std::move(g.weight);
            if (need_b) res[at_w + 1] = std::move(g.bias);
        }
        if (create_graph && grad_output.requires_grad()) {
            // no second derivative: results that say so when they are differentiated
            auto fail = std::make_shared<torch::autograd::DelayedError>(
                "trying to differentiate twice a function that was marked with @once_differentiable", (int64_t)n);
            for (auto& t : res)
                if (t.defined()) t = t.detach().set_requires_grad(true);
            return fail->apply(std::move(res));
        }
        return res;
    }
};

Tensor with_history(const Config& c, const Tensor& out, const Tensor& input, const Tensor& offset, const Tensor& weight, const Tensor& bias) {
    const bool deform = c.cpg > 0;
    const bool any = c10::GradMode::is_enabled() &&
                     (input.requires_grad() || weight.requires_grad() || (deform && offset.requires_grad()) || (bias.defined() && bias.requires_grad()));
    if (!any) return out;
    auto fn = std::shared_ptr<LayerBackward>(new LayerBackward(), torch::autograd::deleteNode);
    fn->cfg = c;
    fn->has_bias = bias.defined();
    fn->input_ = SavedVariable(input, false);
    if (deform) fn->offset_ = SavedVariable(offset, false);
    fn->weight_ = SavedVariable(weight, false);
    torch::autograd::edge_list edges;
    edges.reserve(4);
    edges.push_back(torch::autograd::impl::gradient_edge(input));
    if (deform) edges.push_back(torch::autograd::impl::gradient_edge(offset));
    edges.push_back(torch::autograd::impl::gradient_edge(weight));
    if (bias.defined()) edges.push_back(torch::autograd::impl::gradient_edge(bias));
    // (tensors that need no gradient get no edge)
    const Tensor* ts[4] = {&input, deform ? &offset : &weight, deform ? &weight : &bias, &bias};
    for (size_t i = 0; i < edges.size(); ++i)
        if (!ts[i]->requires_grad()) edges[i] = torch::autograd::Edge();
    fn->set_next_edges(std::move(edges));
    torch::autograd::set_history(out, fn);
    return out;
}

Tensor conv_offset_forward(const Config& c, const Tensor& input, const Tensor& offset, const Tensor& weight, const Tensor& bias) {
    device_check(input, {&offset, &weight, &bias});
    int64_t out[3];
    shape_check(c, input, weight, offset, out);
    const Geometry g = geometry(c, input, weight, out);
    if (bias.defined()) check(bias.dim() == 1 && bias.size(0) == weight.size(0), "bias size");
    c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(input.device());
    const Tensor in = input.contiguous(), off = offset.contiguous(), w = weight.contiguous(), b = bias.defined() ? bias.contiguous() : Tensor();
    int64_t sizes[5] = {input.size(0), weight.size(0), out[0], out[1], c.nd == 3 ? out[2] : 1};
    Tensor output = at::empty(at::IntArrayRef(sizes, c.nd + 2), in.options());
    const Tensor ws = workspace_tensor(in, g.ws_bytes);
    check_rc(run_forward(c.nd, dtype_index(in.scalar_type()), in, w, off, b, output, g.v,
                         workspace(ws, g.ws_bytes, c10::hip::getCurrentHIPStream(in.device().index()).stream())));
    return output;
}

Tensor conv2d_forward(const Config& c, const Tensor& input, const Tensor& weight, const Tensor& bias) {
    int64_t out[3];
    conv_check(c, input, weight, bias, out);
    const Geometry geo = geometry(c, input, weight, out);
    const int* g = geo.v;
    check(geo.ws_bytes > 0, "inconsistent convolution geometry");
    c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(input.device());
    const Tensor in = input.contiguous(), w = weight.contiguous(), b = bias.defined() ? bias.contiguous() : Tensor();
    Tensor output = at::empty({input.size(0), weight.size(0), out[0], out[1]}, in.options());
    const Tensor wst = workspace_tensor(in, geo.ws_bytes);
    const Workspace ws = workspace(wst, geo.ws_bytes, c10::hip::getCurrentHIPStream(in.device().index()).stream());
    check_rc(in.scalar_type() == at::kFloat
                 ? conv2d_forward_f32(cptr<float>(in), cptr<float>(w), cptr<float>(b), mptr<float>(output), GEOC(g), ws.p, ws.n, ws.stream)
                 : conv2d_forward_f64(cptr<double>(in), cptr<double>(w), cptr<double>(b), mptr<double>(output), GEOC(g), ws.p, ws.n, ws.stream));
    return output;
}

// ---- Python entry points -------------------------------------------------------------------
int as_int(PyObject* o) {
    PyObject* i = PyNumber_Long(o);
    if (!i) throw python_error();
    const long v = PyLong_AsLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    if (v > INT32_MAX || v < INT32_MIN) throw std::runtime_error("integer argument out of range");
    return (int)v;
}
void as_ints(PyObject* o, int nd, int* out) {       // one number for all axes, or a sequence of nd
    if (PyLong_Check(o)) {
        for (int a = 0; a < nd; ++a) out[a] = as_int(o);
        return;
    }
    PyObject* s = PySequence_Tuple(o);
    if (!s) throw python_error();
    const Py_ssize_t n = PyTuple_GET_SIZE(s);
    if (n != nd) {
        PyObject* text = PyObject_Repr(s);
        const std::string r = text ? PyUnicode_AsUTF8(text) : "?";
        Py_XDECREF(text);
        Py_DECREF(s);
        throw std::runtime_error("expected " + std::to_string(nd) + " values, got " + r);
    }
    try {
        for (int a = 0; a < nd; ++a) out[a] = as_int(PyTuple_GET_ITEM(s, a));
    } catch (...) {
        Py_DECREF(s);
        throw;
    }
    Py_DECREF(s);
}
Tensor as_tensor(PyObject* o, const char* what, bool optional = false) {
    if (optional && o == Py_None) return Tensor();
    if (!THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "%s must be a tensor, got %s", what, Py_TYPE(o)->tp_name);
        throw python_error();
    }
    return THPVariable_Unpack(o);
}

PyObject* wrap(const Tensor& t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
PyObject* wrap(const Gradients& g, bool deform) {
    const Tensor* ts[4] = {&g.input, deform ? &g.offset : &g.weight, deform ? &g.weight : &g.bias, &g.bias};
    const Py_ssize_t n = deform ? 4 : 3;
    PyObject* r = PyTuple_New(n);
    if (!r) throw python_error();
    for (Py_ssize_t i = 0; i < n; ++i) PyTuple_SET_ITEM(r, i, wrap(*ts[i]));
    return r;
}
// stride, padding, dilation, channel_per_group, group, standard, oob_zero
Config layer_config(int nd, PyObject* const* a) {
    Config c;
    c.nd = nd;
    as_ints(a[0], nd, c.stride);
    as_ints(a[1], nd, c.pad);
    as_ints(a[2], nd, c.dil);
    c.cpg = as_int(a[3]);
    c.group = as_int(a[4]);
    c.standard = PyObject_IsTrue(a[5]) == 1;
    c.oob_zero = PyObject_IsTrue(a[6]) == 1;
    check(c.cpg > 0, "off channel");
    return c;
}
// stride, padding, dilation, group
Config conv_config(PyObject* const* a) {
    Config c;
    c.nd = 2;
    as_ints(a[0], 2, c.stride);
    as_ints(a[1], 2, c.pad);
    as_ints(a[2], 2, c.dil);
    c.group = as_int(a[3]);
    return c;
}
int axes(PyObject* o) {
    const int nd = as_int(o);
    check(nd == 2 || nd == 3, "two or three axes");
    return nd;
}

// Whether a call has to go through PyTorch's Function.apply, because more than backward has to know about it:
// - a trace being recorded: the tracer sees no operator of libdcn_amd.so and would keep the allocation of the output alone;
// - an argument with a forward-mode tangent, which the node here would drop without a word (Function.apply refuses it);
// - functorch transforms (vmap, torch.func.grad, ...), likewise refused there, and wrappers that outlived one.
bool wants_function(std::initializer_list<const Tensor*> args) {
    using c10::DispatchKey;
    using c10::DispatchKeySet;
    if (torch::jit::tracer::isTracing()) return true;
    if (c10::impl::tls_local_dispatch_key_set().included_.has_any(
            DispatchKeySet({DispatchKey::FuncTorchDynamicLayerFrontMode, DispatchKey::FuncTorchDynamicLayerBackMode})))
        return true;
    for (const Tensor* t : args)
        if (t->defined() && (t->_fw_grad(0).defined() ||
                             t->key_set().has_any(DispatchKeySet({DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched}))))
            return true;
    return false;
}
PyObject* py_wants_function(PyObject*, PyObject* arg) {
    HANDLE_TH_ERRORS
    const Tensor t = as_tensor(arg, "argument");
    return PyBool_FromLong(wants_function({&t}));
    END_HANDLE_TH_ERRORS
}

// conv_offset(nd, inputs, offset, weight, bias, stride, padding, dilation, channel_per_group, group, standard, oob_zero):
// the layer with its backward node; NotImplemented when the call has to go through Function.apply
template <bool HISTORY> PyObject* py_conv_offset(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    check(n == 12, "conv_offset takes 12 arguments");
    const int nd = axes(a[0]);
    const Tensor input = as_tensor(a[1], "inputs"), offset = as_tensor(a[2], "offset"), weight = as_tensor(a[3], "weight"), bias = as_tensor(a[4], "bias", true);
    if (HISTORY && wants_function({&input, &offset, &weight, &bias})) Py_RETURN_NOTIMPLEMENTED;
    const Config c = layer_config(nd, a + 5);
    Tensor out;
    {
        pybind11::gil_scoped_release nogil;
        out = conv_offset_forward(c, input, offset, weight, bias);
        if (HISTORY) out = with_history(c, out, input, offset, weight, bias);
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}
// conv_offset_backward(nd, inputs, offset, weight, grad_output, stride, padding, dilation, channel_per_group, group, standard,
// oob_zero, need_data, need_weight, need_bias): the gradients of inputs, offset, weight, bias, None where not needed
PyObject* py_conv_offset_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    check(n == 15, "conv_offset_backward takes 15 arguments");
    const int nd = axes(a[0]);
    const Tensor input = as_tensor(a[1], "inputs"), offset = as_tensor(a[2], "offset"), weight = as_tensor(a[3], "weight"), go = as_tensor(a[4], "grad_output");
    const Config c = layer_config(nd, a + 5);
    const bool data = PyObject_IsTrue(a[12]) == 1, w = PyObject_IsTrue(a[13]) == 1, b = PyObject_IsTrue(a[14]) == 1;
    Gradients g;
    {
        pybind11::gil_scoped_release nogil;
        c10::AutoGradMode no_grad(false);
        const c10::OptionalDeviceGuard guard(input.device());
        g = conv_offset_backward(c, input, offset, weight, go, data, w, b);
    }
    return wrap(g, true);
    END_HANDLE_TH_ERRORS
}
// conv2d(inputs, weight, bias, stride, padding, dilation, group): the layer with its backward node, or NotImplemented
template <bool HISTORY> PyObject* py_conv2d(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    check(n == 7, "conv2d takes 7 arguments");
    const Tensor input = as_tensor(a[0], "inputs"), weight = as_tensor(a[1], "weight"), bias = as_tensor(a[2], "bias", true);
    if (HISTORY && wants_function({&input, &weight, &bias})) Py_RETURN_NOTIMPLEMENTED;
    const Config c = conv_config(a + 3);
    Tensor out;
    {
        pybind11::gil_scoped_release nogil;
        out = conv2d_forward(c, input, weight, bias);
        if (HISTORY) out = with_history(c, out, input, Tensor(), weight, bias);
    }
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}
// conv2d_backward(inputs, weight, grad_output, stride, padding, dilation, group, need_data, need_weight, need_bias)
PyObject* py_conv2d_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    check(n == 10, "conv2d_backward takes 10 arguments");
    const Tensor input = as_tensor(a[0], "inputs"), weight = as_tensor(a[1], "weight"), go = as_tensor(a[2], "grad_output");
    const Config c = conv_config(a + 3);
    const bool data = PyObject_IsTrue(a[7]) == 1, w = PyObject_IsTrue(a[8]) == 1, b = PyObject_IsTrue(a[9]) == 1;
    Gradients g;
    {
        pybind11::gil_scoped_release nogil;
        c10::AutoGradMode no_grad(false);
        const c10::OptionalDeviceGuard guard(input.device());
        g = conv2d_backward(c, input, weight, go, data, w, b);
    }
    return wrap(g, false);
    END_HANDLE_TH_ERRORS
}
// shape_check(nd, inputs, weight, offset, output_shape, stride, padding, dilation, channel_per_group, group, standard)
PyObject* py_shape_check(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    check(n == 11, "shape_check takes 11 arguments");
    Config c;
    c.nd = axes(a[0]);
    const Tensor input = as_tensor(a[1], "inputs"), weight = as_tensor(a[2], "weight"), offset = as_tensor(a[3], "offset");
    std::vector<int64_t> sizes;
    for (const auto& v : pybind11::reinterpret_borrow<pybind11::sequence>(a[4])) sizes.push_back(v.cast<int64_t>());
    as_ints(a[5], c.nd, c.stride);
    as_ints(a[6], c.nd, c.pad);
    as_ints(a[7], c.nd, c.dil);
    c.cpg = as_int(a[8]);
    c.group = as_int(a[9]);
    c.standard = PyObject_IsTrue(a[10]) == 1;
    const at::IntArrayRef shape(sizes);
    int64_t out[3];
    shape_check(c, input, weight, offset, out, &shape);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}
// set_error(type): the exception class for calls that the library rejects
PyObject* py_set_error(PyObject*, PyObject* type) {
    Py_INCREF(type);
    Py_XDECREF(g_library_error);
    g_library_error = type;
    Py_RETURN_NONE;
}

using FastCall = PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t);
PyCFunction method(FastCall f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }
PyMethodDef methods[] = {{"conv_offset", method(py_conv_offset<true>), METH_FASTCALL, nullptr},
                         {"conv_offset_forward", method(py_conv_offset<false>), METH_FASTCALL, nullptr},
                         {"conv_offset_backward", method(py_conv_offset_backward), METH_FASTCALL, nullptr},
                         {"conv2d", method(py_conv2d<true>), METH_FASTCALL, nullptr},
                         {"conv2d_forward", method(py_conv2d<false>), METH_FASTCALL, nullptr},
                         {"conv2d_backward", method(py_conv2d_backward), METH_FASTCALL, nullptr},
                         {"wants_function", py_wants_function, METH_O, nullptr},
                         {"shape_check", method(py_shape_check), METH_FASTCALL, nullptr},
                         {"set_error", py_set_error, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module_def); }
