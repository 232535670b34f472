// C ABI of libdcn_amd.so (declared in include/dcn_amd.h).  No device memory is allocated here and
// nothing synchronises; all work is enqueued on the caller's stream.
#include "dcn_host.h"
#include "dcn_forward.h"

namespace {

using namespace dcn;

// ---------------------------------------------------------------------------------------------
// Mixed precision: tensors stored as bfloat16 / binary16, accumulation in float32.  Each call first
// offers the layer to the kernel that reads the 16-bit tensors itself and multiplies on the 16-bit
// matrix instructions (float results in a float copy at the front of the workspace, rounded once
// when they are written back); where that kernel declines, the tensors are widened into float
// copies at the front of the workspace and the float32 kernels run on them with the rest of it.
struct Carver {
    char* p;
    size_t left;
    float* take(size_t n) {
        const size_t b = align256(n * sizeof(float));
        if (!p || b > left) return nullptr;
        float* r = reinterpret_cast<float*>(p);
        p += b;
        left -= b;
        return r;
    }
};
template <typename S> int widen(const S* src, float* dst, size_t n, hipStream_t s) {
    const unsigned blocks = (unsigned)((n + 1023) / 1024 > 8192 ? 8192 : (n + 1023) / 1024);
    hipLaunchKernelGGL(widen_kernel<S>, dim3(blocks ? blocks : 1), dim3(256), 0, s, src, dst, n);
    return check_launch("widen_kernel");
}
template <typename S> int narrow(const float* src, S* dst, size_t n, hipStream_t s) {
    const unsigned blocks = (unsigned)((n + 1023) / 1024 > 8192 ? 8192 : (n + 1023) / 1024);
    hipLaunchKernelGGL(narrow_kernel<S>, dim3(blocks ? blocks : 1), dim3(256), 0, s, src, dst, n);
    return check_launch("narrow_kernel");
}
struct Sizes16 { size_t in, w, off, out; };
Sizes16 sizes16(const Params& P, int nd) {
    return Sizes16{(size_t)P.N * P.C_in * P.inV, (size_t)P.C_out * P.Cg * P.kV, (size_t)P.N * P.DG * P.kV * nd * P.outV,
                   (size_t)P.N * P.C_out * P.outV};
}
// float copies of every tensor any of the three calls touches (nd = 3 bounds the offsets of either operator)
size_t copies16_bytes(int N, int C_in, int C_out, size_t inV, size_t outV, int kV, int G, int cpg) {
    const size_t in = (size_t)N * C_in * inV, w = (size_t)C_out * (C_in / G) * kV, off = (size_t)N * (C_in / cpg) * kV * 3 * outV,
                 out = (size_t)N * C_out * outV;
    return 2 * align256(in * 4) + 2 * align256(w * 4) + 2 * align256(off * 4) + align256(out * 4) + align256((size_t)C_out * 4);
}

// grad_weight alone, added to what it holds (plain: no offsets)
template <typename T, int ND>
int backward_weight(const Geometry& g, const T* in, const T* off, const T* gout, T* gw, void* ws, size_t ws_bytes, hipStream_t s, bool plain = false) {
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || (!off && !plain) || !gout || !gw) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    WeightCall<T, T> call;
    Prep prep;
    const PlanChoice none = {};
    if (int rc = backward_weight_plan<T, ND, T>(P, in, off, gout, ws, ws_bytes, false, call, prep, nullptr)) return rc;
    if (int rc = launch_prepare<T, T>(P, none, prep, static_cast<const T*>(nullptr), off, 0, s)) return rc;
    return backward_weight_run<T, ND, T>(call, off, gw, nullptr, true, s);
}

template <typename S, int ND>
int forward16(const Geometry& g, const S* in, const S* w, const S* off, const S* bias, S* out, void* ws, size_t ws_bytes,
              hipStream_t s) {
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !w || !off || !out) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    if (native16()) {       // the LDS-halo kernel reads the 16-bit tensors itself and multiplies with 16-bit matrix instructions
        bool declined = false;
        if (int rc = forward<float, ND, S>(g, in, w, off, bias, out, ws, ws_bytes, s, &declined)) return rc;
        if (!declined) return DCN_OK;
    }
    const Sizes16 z = sizes16(P, ND);
    Carver c{static_cast<char*>(ws), ws ? ws_bytes : 0};
    float *fin = c.take(z.in), *fw = c.take(z.w), *foff = c.take(z.off), *fout = c.take(z.out), *fb = bias ? c.take(P.C_out) : nullptr;
    if (!fin || !fw || !foff || !fout || (bias && !fb)) return fail(DCN_E_WORKSPACE, "workspace too small");
    if (int rc = widen(in, fin, z.in, s)) return rc;
    if (int rc = widen(w, fw, z.w, s)) return rc;
    if (int rc = widen(off, foff, z.off, s)) return rc;
    if (bias) if (int rc = widen(bias, fb, (size_t)P.C_out, s)) return rc;
    if (int rc = forward<float, ND>(g, fin, fw, foff, fb, fout, c.p, c.left, s)) return rc;
    return narrow(fout, out, z.out, s);
}
template <typename S, int ND>
int backward_input_offset16(const Geometry& g, const S* in, const S* w, const S* off, const S* gout, S* gin, S* goff, void* ws,
                            size_t ws_bytes, hipStream_t s) {
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !w || !off || !gout || !gin || !goff) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    const Sizes16 z = sizes16(P, ND);
    Carver c{static_cast<char*>(ws), ws ? ws_bytes : 0};
    float *fin = c.take(z.in), *fw = c.take(z.w), *foff = c.take(z.off), *fgout = c.take(z.out), *fgin = c.take(z.in), *fgoff = c.take(z.off);
    if (!fin || !fw || !foff || !fgout || !fgin || !fgoff) return fail(DCN_E_WORKSPACE, "workspace too small");
    if (int rc = widen(gin, fgin, z.in, s)) return rc;            // grad_input is accumulated into
    // the fused kernel reads the 16-bit tensors itself and forms the grad columns with 16-bit matrix
    // instructions (the products of 16-bit values are exact in float, so the results are those of the
    // float32 kernel up to the order of the sums); the gradients leave it as float and are rounded once
    bool declined = true;
    if (native16()) {
        declined = false;
        if (int rc = backward_input_offset<float, ND, S>(g, in, w, off, gout, fgin, fgoff, c.p, c.left, s, 0, &declined)) return rc;
    }
    if (declined) {
        if (int rc = widen(in, fin, z.in, s)) return rc;
        if (int rc = widen(w, fw, z.w, s)) return rc;
        if (int rc = widen(off, foff, z.off, s)) return rc;
        if (int rc = widen(gout, fgout, z.out, s)) return rc;
        if (int rc = backward_input_offset<float, ND>(g, fin, fw, foff, fgout, fgin, fgoff, c.p, c.left, s)) return rc;
    }
    if (int rc = narrow(fgin, gin, z.in, s)) return rc;
    return narrow(fgoff, goff, z.off, s);
}
template <typename S, int ND>
int backward_weight16(const Geometry& g, const S* in, const S* off, const S* gout, S* gw, void* ws, size_t ws_bytes, hipStream_t s) {
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !off || !gout || !gw) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    const Sizes16 z = sizes16(P, ND);
    Carver c{static_cast<char*>(ws), ws ? ws_bytes : 0};
    float *fin = c.take(z.in), *foff = c.take(z.off), *fgout = c.take(z.out), *fgw = c.take(z.w);
    if (!fin || !foff || !fgout || !fgw) return fail(DCN_E_WORKSPACE, "workspace too small");
    if (int rc = widen(gw, fgw, z.w, s)) return rc;               // grad_weight is accumulated into
    bool declined = true;
    if (native16()) {
        WeightCall<float, S> call;
        Prep prep;
        const PlanChoice none = {};
        if (int rc = backward_weight_plan<float, ND, S>(P, in, off, gout, c.p, c.left, false, call, prep, &declined)) return rc;
        if (!declined) {
            if (int rc = launch_prepare<float, S>(P, none, prep, static_cast<const S*>(nullptr), off, 0, s)) return rc;
            if (int rc = backward_weight_run<float, ND, S>(call, off, fgw, nullptr, true, s)) return rc;
        }
    }
    if (declined) {
        if (int rc = widen(in, fin, z.in, s)) return rc;
        if (int rc = widen(off, foff, z.off, s)) return rc;
        if (int rc = widen(gout, fgout, z.out, s)) return rc;
        if (int rc = backward_weight<float, ND>(g, fin, foff, fgout, fgw, c.p, c.left, s)) return rc;
    }
    return narrow(fgw, gw, z.w, s);
}

// ---------------------------------------------------------------------------------------------
// The backward pass of a layer in one call: the gradients asked for (null: not wanted), written, not
// added.  What the operators need beforehand -- cleared buffers, packed weights, channels-last copies,
// the sums for grad_bias -- is one launch (backward_prepare_kernel).
// Workspace: see LayerNeed.
template <typename S> struct Wide { typedef float type; };
template <> struct Wide<double> { typedef double type; };
template <typename S>
__global__ __launch_bounds__(256) void narrow_gradients_kernel(const float* __restrict__ a, S* __restrict__ da, size_t na, const float* __restrict__ b,
                                                               S* __restrict__ db, size_t nb, const float* __restrict__ c, S* __restrict__ dc, size_t nc,
                                                               const float* __restrict__ d, S* __restrict__ dd, size_t nd, bool octets, int N, int C,
                                                               unsigned V) {
    const size_t step = (size_t)gridDim.x * 256, first = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (octets) octets_to_planes(a, N, C, V, false, first, step, [&](size_t to, float v) { da[to] = S::narrow(v); });
    else
        for (size_t i = first; i < na; i += step) da[i] = S::narrow(a[i]);
    for (size_t i = first; i < nb; i += step) db[i] = S::narrow(b[i]);
    for (size_t i = first; i < nc; i += step) dc[i] = S::narrow(c[i]);
    for (size_t i = first; i < nd; i += step) dd[i] = S::narrow(d[i]);
}
template <typename S, int ND>
int layer_backward(const Geometry& g, const S* in, const S* w, const S* off, const S* gout, S* gin, S* goff, S* gw, S* gb, void* ws, size_t ws_bytes,
                   hipStream_t s, unsigned flags) {
    typedef typename Wide<S>::type T;
    constexpr bool S16 = !std::is_same<S, T>::value;
    Params P;
    if (int rc = validate(g, P)) return rc;
    const bool data = gin || goff;
    if (!in || !w || !off || !gout || (data && (!gin || !goff)) || (gb && !gw)) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    const Sizes16 z = sizes16(P, ND);
    char* p = static_cast<char*>(ws);
    size_t left = ws ? ws_bytes : 0;
    auto take = [&](size_t bytes) -> void* {
        bytes = align256(bytes);
        if (bytes > left) return nullptr;
        void* r = p;
        p += bytes;
        left -= bytes;
        return r;
    };
    T *tgin, *tgoff, *tgw, *tgb;
    if constexpr (S16) {
        tgin = data ? static_cast<T*>(take(z.in * 4)) : nullptr;
        tgoff = data ? static_cast<T*>(take(z.off * 4)) : nullptr;
        tgw = gw ? static_cast<T*>(take(z.w * 4)) : nullptr;
        tgb = gb ? static_cast<T*>(take((size_t)P.C_out * 4)) : nullptr;
        if ((data && (!tgin || !tgoff)) || (gw && !tgw) || (gb && !tgb)) return fail(DCN_E_WORKSPACE, "workspace too small");
    } else {
        tgin = gin; tgoff = goff; tgw = gw; tgb = gb;
    }
    const LayerNeed need = layer_need<T, S>(ND, P.N, P.C_in, P.C_out, P.inV, P.outV, P.kV, P.G, P.cpg);
    char* const shared = p;                             // (the float copies below lie here, too)
    const size_t shared_bytes = left;
    void *dws = data ? take(need.data) : nullptr, *wws = gw ? take(need.weight) : nullptr;
    if ((data && !dws) || (gw && !wws)) return fail(DCN_E_WORKSPACE, "workspace too small");
    Prep prep;
    WeightCall<T, S> call;
    const PlanChoice none = {};
    // (16-bit storage: the kernels that read it may decline a layer, which then runs on widened copies)
    bool wdeclined = S16 && !native16(), ddeclined = wdeclined;
    if (gw && !wdeclined)
        if (int rc = backward_weight_plan<T, ND, S>(P, in, off, gout, wws, need.weight, gb != nullptr, call, prep, S16 ? &wdeclined : nullptr)) return rc;
    if (data && !ddeclined)
        if (int rc = backward_input_offset<T, ND, S>(g, in, w, off, gout, tgin, tgoff, dws, need.data, s, flags, S16 ? &ddeclined : nullptr, &prep)) return rc;
    if (data && ddeclined) prep.zero(tgin, z.in * sizeof(T));      // (else the operator sees to it)
    if (!data || ddeclined)
        if (int rc = launch_prepare<T, S>(P, none, prep, w, off, 0, s)) return rc;
    if (gw && !wdeclined)
        if (int rc = backward_weight_run<T, ND, S>(call, off, tgw, tgb, false, s)) return rc;
    bool narrowed = false;                              // grad_input
    if constexpr (S16) {
        const bool wide_data = data && ddeclined, wide_weight = gw && wdeclined;
        if (wide_weight && prep.octets) {               // they lie where the copies go
            const unsigned blocks = (unsigned)((z.in + 1023) / 1024 > 8192 ? 8192 : (z.in + 1023) / 1024);
            hipLaunchKernelGGL(narrow_gradients_kernel<S>, dim3(blocks), dim3(256), 0, s, prep.octets, gin, z.in, nullptr, nullptr, 0, nullptr, nullptr, 0, nullptr,
                               nullptr, 0, true, P.N, P.C_in, P.inV);
            if (int rc = check_launch("narrow_gradients_kernel")) return rc;
            if (trace_plans()) fprintf(stderr, "dcn layer_backward: grad_input rounded ahead of the widened copies\n");
            prep.octets = nullptr;
            narrowed = true;
        }
        if (wide_data || wide_weight) {
            p = shared;                                 // the kernels above are done with their operands by the time the next ones run
            left = shared_bytes;
            float* copy[4] = {static_cast<float*>(take(z.in * 4)), static_cast<float*>(take(z.w * 4)), static_cast<float*>(take(z.off * 4)), static_cast<float*>(take(z.out * 4))};
            void* ops = take(need.wide);
            if (!copy[0] || !copy[1] || !copy[2] || !copy[3] || !ops) return fail(DCN_E_WORKSPACE, "workspace too small");
            if (int rc = widen(in, copy[0], z.in, s)) return rc;
            if (int rc = widen(w, copy[1], z.w, s)) return rc;
            if (int rc = widen(off, copy[2], z.off, s)) return rc;
            if (int rc = widen(gout, copy[3], z.out, s)) return rc;
            const T *fin = copy[0], *fw = copy[1], *foff = copy[2], *fgout = copy[3];
            if (wide_data)
                if (int rc = backward_input_offset<T, ND>(g, fin, fw, foff, fgout, tgin, tgoff, ops, need.wide, s, flags)) return rc;
            if (wide_weight) {
                WeightCall<T, T> wide;
                Prep wprep;
                if (int rc = backward_weight_plan<T, ND, T>(P, fin, foff, fgout, ops, need.weight, gb != nullptr, wide, wprep, nullptr)) return rc;
                if (int rc = launch_prepare<T, T>(P, none, wprep, fw, foff, 0, s)) return rc;
                if (int rc = backward_weight_run<T, ND, T>(wide, foff, tgw, tgb, false, s)) return rc;
            }
        }
    }
    if constexpr (S16) {
        const size_t na = data && !narrowed ? z.in : 0, nb = data ? z.off : 0, nc = gw ? z.w : 0, nd = gb ? (size_t)P.C_out : 0, most = na + nb + nc;
        const unsigned blocks = (unsigned)((most + 1023) / 1024 > 8192 ? 8192 : (most + 1023) / 1024 + 1);
        hipLaunchKernelGGL(narrow_gradients_kernel<S>, dim3(blocks), dim3(256), 0, s, prep.octets ? prep.octets : (const float*)tgin, gin, na, (const float*)tgoff, goff, nb, (const float*)tgw, gw,
                           nc, (const float*)tgb, gb, nd, prep.octets != nullptr, P.N, P.C_in, P.inV);
        return check_launch("narrow_gradients_kernel");
    }
    return DCN_OK;
}

// ---------------------------------------------------------------------------------------------
// Plain 2-D convolution: the reference's conv2d package (conv2d/lib/conv2d_cuda.cpp:77-290, kernels
// conv2d/lib/conv2d_cuda_kernel.cu:25-169: im2col / col2im with integer taps and one GEMM per sample
// and group).  It is the 2-D deformable layer with every offset zero, one deformable group and the
// dilation-aware output size (conv2d/lib/conv2d_cuda.cpp:20-22).  The float32 forward pass, which is also the
// backward pass to the input at stride 1, has a kernel of its own where that is faster (plain_conv_kernel); the rest
// runs on the deformable layer's: a null offset means zeros to the float32 forward pass and to the backward
// pass to the weight; the others get a zero offset tensor at the front of the workspace, behind it scratch for the
// grad_offset that one fallback kernel of backward-to-input writes, then the deformable layer's own workspace.
template <typename T> size_t conv2d_zero_bytes(int N, int kV, size_t outV) { return align256((size_t)N * 2 * kV * outV * sizeof(T)); }
template <typename T>
int conv2d_offsets(const Geometry& g, void* ws, size_t ws_bytes, hipStream_t s, T** off, T** scratch, void** rest, size_t* rest_bytes) {
    if (g.N <= 0 || g.out[1] <= 0 || g.out[2] <= 0 || g.k[1] <= 0 || g.k[2] <= 0) return fail(DCN_E_ARGUMENT, "batch / output / kernel extents must be positive");
    const size_t zb = conv2d_zero_bytes<T>(g.N, g.k[1] * g.k[2], (size_t)g.out[1] * g.out[2]);
    if (!ws || ws_bytes < 2 * zb) return fail(DCN_E_WORKSPACE, "workspace too small");
    *off = static_cast<T*>(ws);
    *scratch = reinterpret_cast<T*>(static_cast<char*>(ws) + zb);
    *rest = static_cast<char*>(ws) + 2 * zb;
    *rest_bytes = ws_bytes - 2 * zb;
    const size_t n = zb / sizeof(T);
    const unsigned blocks = (unsigned)((n + 1023) / 1024 > 4096 ? 4096 : (n + 1023) / 1024);
    hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(blocks), dim3(256), 0, s, *off, n);
    return check_launch("fill_zero_kernel");
}
template <typename T>
int conv2d_forward(Geometry g, const T* in, const T* w, const T* bias, T* out, void* ws, size_t ws_bytes, hipStream_t s) {
    g.cpg = g.C_in;
    if constexpr (sizeof(T) == 4) {
        bool declined = false;
        if (int rc = forward<T, 2>(g, in, w, static_cast<const T*>(nullptr), bias, out, ws, ws_bytes, s, &declined)) return rc;
        if (!declined) return DCN_OK;
    }
    T *off, *scratch; void* rest; size_t rest_bytes;
    if (int rc = conv2d_offsets<T>(g, ws, ws_bytes, s, &off, &scratch, &rest, &rest_bytes)) return rc;
    return forward<T, 2>(g, in, w, off, bias, out, rest, rest_bytes, s);
}
template <typename T>
int conv2d_backward_input(Geometry g, const T* w, const T* gout, T* gin, void* ws, size_t ws_bytes, hipStream_t s) {
    g.cpg = g.C_in;
    T *off, *scratch; void* rest; size_t rest_bytes;
    if (int rc = conv2d_offsets<T>(g, ws, ws_bytes, s, &off, &scratch, &rest, &rest_bytes)) return rc;
    return backward_input_offset<T, 2>(g, static_cast<const T*>(nullptr), w, static_cast<const T*>(off), gout, gin, scratch, rest, rest_bytes, s, FLAG_INPUT_ONLY);
}
template <typename T>
int conv2d_backward_weight(Geometry g, const T* in, const T* gout, T* gw, void* ws, size_t ws_bytes, hipStream_t s) {
    g.cpg = g.C_in;
    return backward_weight<T, 2>(g, in, static_cast<const T*>(nullptr), gout, gw, ws, ws_bytes, s, true);
}
// The gradients asked for (null: not wanted), written.  grad_input of a layer of stride 1 is a
// convolution itself -- grad_output with the weight's channels exchanged and its taps in reverse, padded
// by dilation * (k - 1) - pad -- and runs as a forward pass: no scatter (64 -> 64 channels, 8 x 56 x 56: 26 us
// against 146 for the kernel that adds up grad_input in LDS).
template <typename T>
int conv2d_layer_backward(Geometry g, const T* in, const T* w, const T* gout, T* gin, T* gw, T* gb, void* ws, size_t ws_bytes, hipStream_t s) {
    g.cpg = g.C_in;
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !w || !gout || (gb && !gw)) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    const size_t wbytes = align256(backward_weight_need<T>(P.N, P.C_in, P.C_out, P.inV, P.outV, P.kV, P.G));
    if (!ws || ws_bytes < wbytes) return fail(DCN_E_WORKSPACE, "workspace too small");
    if (gin) {
        void* dws = static_cast<char*>(ws) + wbytes;
        bool done = false;
        if constexpr (sizeof(T) == 4) {
            Geometry t = g;
            bool fits = true;
            t.C_in = t.cpg = g.C_out;
            t.C_out = g.C_in;
            for (int a = 1; a < 3; ++a) {
                t.in[a] = g.out[a];
                t.out[a] = g.in[a];
                t.pad[a] = g.dil[a] * (g.k[a] - 1) - g.pad[a];
                fits = fits && g.stride[a] == 1 && t.pad[a] >= 0;
            }
            if (fits) {
                bool declined = false;
                if (int rc = forward<T, 2>(t, gout, w, static_cast<const T*>(nullptr), static_cast<const T*>(nullptr), gin, dws, ws_bytes - wbytes, s, &declined, true)) return rc;
                done = !declined;
            }
        }
        if (!done) {
            const size_t n = (size_t)P.N * P.C_in * P.inV;
            const unsigned blocks = (unsigned)((n + 1023) / 1024 > 4096 ? 4096 : (n + 1023) / 1024);
            hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(blocks), dim3(256), 0, s, gin, n);
            if (int rc = check_launch("fill_zero_kernel")) return rc;
            if (int rc = conv2d_backward_input<T>(g, w, gout, gin, dws, ws_bytes - wbytes, s)) return rc;
        }
    }
    if (!gw) return DCN_OK;
    WeightCall<T, T> call;
    Prep prep;
    const PlanChoice none = {};
    const T* off = nullptr;
    if (int rc = backward_weight_plan<T, 2, T>(P, in, off, gout, ws, wbytes, gb != nullptr, call, prep, nullptr)) return rc;
    if (int rc = launch_prepare<T, T>(P, none, prep, w, off, 0, s)) return rc;
    return backward_weight_run<T, 2, T>(call, off, gw, gb, false, s);
}

Geometry geo3(int batch, int input_c, int output_c, int input_l, int input_h, int input_w, int output_l,
              int output_h, int output_w, int kernel_l, int kernel_h, int kernel_w, int pad_l, int pad_h,
              int pad_w, int stride_l, int stride_h, int stride_w, int dilation_l, int dilation_h,
              int dilation_w, int cpg, int group) {
    return Geometry{3, batch, input_c, output_c, {input_l, input_h, input_w}, {output_l, output_h, output_w},
                    {kernel_l, kernel_h, kernel_w}, {pad_l, pad_h, pad_w}, {stride_l, stride_h, stride_w},
                    {dilation_l, dilation_h, dilation_w}, cpg, group};
}
Geometry geo2(int batch, int input_c, int output_c, int input_h, int input_w, int output_h, int output_w,
              int kernel_h, int kernel_w, int pad_h, int pad_w, int stride_h, int stride_w, int dilation_h,
              int dilation_w, int cpg, int group) {
    return Geometry{2, batch, input_c, output_c, {1, input_h, input_w}, {1, output_h, output_w},
                    {1, kernel_h, kernel_w}, {0, pad_h, pad_w}, {1, stride_h, stride_w},
                    {1, dilation_h, dilation_w}, cpg, group};
}

// ---------------------------------------------------------------------------------------------
// Scratch of the allocation-free entry point: the re-laid-out weight of one forward call.  A
// file-scope device array, so every GPU the library runs on holds NOALLOC_ARRAY_BYTES of it
// until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress: the device address is looked up once per device and kept, and host code
// passes that address, never the name, to kernels.
static __device__ __align__(256) unsigned char scratch[NOALLOC_ARRAY_BYTES];

std::mutex g_scratch_lock;
void* g_scratch_ptr[MAX_DEVICES] = {};

int scratch_address(void** out) {
    int dev = -1;
    if (int rc = device_info(nullptr, &dev)) return rc;
    std::lock_guard<std::mutex> lock(g_scratch_lock);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            g_err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return DCN_E_DEVICE;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return DCN_OK;
}

}  // namespace

#define G3_ARGS batch, input_c, output_c, input_l, input_h, input_w, output_l, output_h, output_w, kernel_l, \
                kernel_h, kernel_w, pad_l, pad_h, pad_w, stride_l, stride_h, stride_w, dilation_l, dilation_h, \
                dilation_w, channel_per_deformable_group, group
#define G2_ARGS batch, input_c, output_c, input_h, input_w, output_h, output_w, kernel_h, kernel_w, pad_h, pad_w, \
                stride_h, stride_w, dilation_h, dilation_w, channel_per_deformable_group, group

extern "C" {

int dcn_version(void) { return 1; }
const char* dcn_arch(void) { return "gfx950"; }
const char* dcn_last_error(void) { return g_err.c_str(); }

size_t dcn_workspace_bytes(int elem_size, int batch, int input_c, int output_c, size_t input_volume,
                           size_t output_volume, int kernel_volume, int group) {
    if (group <= 0 || batch <= 0 || input_c <= 0 || output_c <= 0 || kernel_volume <= 0 || input_volume == 0 ||
        output_volume == 0 || elem_size == 2)      // 16-bit storage: dcn_workspace_bytes_for
        return 0;
    return elem_size == 8
               ? workspace_need<double>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group)
               : workspace_need<float>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group);
}

size_t dcn_workspace_bytes_for(int elem_size, int batch, int input_c, int output_c, size_t input_volume,
                               size_t output_volume, int kernel_volume, int group, int channel_per_deformable_group) {
    if (group <= 0 || batch <= 0 || input_c <= 0 || output_c <= 0 || kernel_volume <= 0 || input_volume == 0 ||
        output_volume == 0 || channel_per_deformable_group <= 0 || input_c % channel_per_deformable_group)
        return 0;
    const int cpg = channel_per_deformable_group;
    if (elem_size == 2)     // bfloat16 / binary16 storage: float copies of the tensors + the float32 workspace
        return copies16_bytes(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group, cpg) +
               workspace_need<float>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group, cpg);
    return elem_size == 8
               ? workspace_need<double>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group, cpg)
               : workspace_need<float>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group, cpg);
}

size_t dcn_layer_backward_workspace_bytes(int elem_size, int nd, int batch, int input_c, int output_c, size_t input_volume, size_t output_volume,
                                          int kernel_volume, int group, int channel_per_deformable_group) {
    if (group <= 0 || batch <= 0 || input_c <= 0 || output_c <= 0 || kernel_volume <= 0 || input_volume == 0 || output_volume == 0 ||
        channel_per_deformable_group <= 0 || input_c % channel_per_deformable_group || input_c % group || output_c % group || nd < 2 || nd > 3)
        return 0;
    const int cpg = channel_per_deformable_group;
#define LAYER_BYTES(T, S) layer_bytes(layer_need<T, S>(nd, batch, input_c, output_c, input_volume, output_volume, kernel_volume, group, cpg))
    return elem_size == 8 ? LAYER_BYTES(double, double) : elem_size == 2 ? LAYER_BYTES(float, Bf16) : LAYER_BYTES(float, float);
#undef LAYER_BYTES
}

int dcn_layer_backward(int nd, int dtype, const void* input, const void* weight, const void* offset, const void* grad_output, void* grad_input, void* grad_offset,
                       void* grad_weight, void* grad_bias, const int* geometry, void* workspace, size_t workspace_bytes, void* stream, unsigned flags) {
    if (!geometry || (nd != 2 && nd != 3)) return fail(DCN_E_ARGUMENT, "two or three axes and their geometry");
    if (flags & ~(unsigned)DCN_FLAG_OOB_OFFSET_GRAD_ZERO) return fail(DCN_E_ARGUMENT, "unknown flag");
    if (flags && dtype >= 2) return fail(DCN_E_ARGUMENT, "oob_offset_grad='zero' is available in float32 and float64 only");
    const int* v = geometry;
    Geometry g{nd, v[0], v[1], v[2], {1, 1, 1}, {1, 1, 1}, {1, 1, 1}, {0, 0, 0}, {1, 1, 1}, {1, 1, 1}, 0, 0};
    v += 3;
    for (int* axis : {g.in, g.out, g.k, g.pad, g.stride, g.dil})
        for (int a = 3 - nd; a < 3; ++a) axis[a] = *v++;
    g.cpg = v[0];
    g.G = v[1];
#define LAYER(S, ND)                                                                                                                              \
    layer_backward<S, ND>(g, (const S*)input, (const S*)weight, (const S*)offset, (const S*)grad_output, (S*)grad_input, (S*)grad_offset,         \
                          (S*)grad_weight, (S*)grad_bias, workspace, workspace_bytes, static_cast<hipStream_t>(stream), flags)
    switch (dtype) {
        case 0: return nd == 3 ? LAYER(float, 3) : LAYER(float, 2);
        case 1: return nd == 3 ? LAYER(double, 3) : LAYER(double, 2);
        case 2: return nd == 3 ? LAYER(Bf16, 3) : LAYER(Bf16, 2);
        case 3: return nd == 3 ? LAYER(Fp16, 3) : LAYER(Fp16, 2);
        default: return fail(DCN_E_ARGUMENT, "unknown data type");
    }
#undef LAYER
}

int dcn3d_forward_noalloc_f32(const float* input, const float* weight, const float* offset, const float* bias,
                              float* output, DCN3D_GEOMETRY, void* stream) {
    const Geometry g = geo3(G3_ARGS);
    Params P;
    if (int rc = validate(g, P)) return rc;
    const size_t need = noalloc_weight_bytes(P);
    if (need > DCN_NOALLOC_SCRATCH_BYTES) {
        char msg[200];
        snprintf(msg, sizeof msg, "layer too large for the allocation-free entry point: its re-laid-out weight takes %zu bytes, "
                 "the fixed scratch holds %zu", need, (size_t)DCN_NOALLOC_SCRATCH_BYTES);
        return fail(DCN_E_WORKSPACE, msg);
    }
    void* ws = nullptr;
    if (int rc = scratch_address(&ws)) return rc;
    return forward<float, 3>(g, input, weight, offset, bias, output, ws, NOALLOC_ARRAY_BYTES,
                             static_cast<hipStream_t>(stream));
}

#define DEFINE_OPS(SUF, T)                                                                                          \
    int dcn3d_forward_##SUF(const T* input, const T* weight, const T* offset, const T* bias, T* output,             \
                            DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {                \
        return forward<T, 3>(geo3(G3_ARGS), input, weight, offset, bias, output, workspace, workspace_bytes,        \
                             static_cast<hipStream_t>(stream));                                                     \
    }                                                                                                               \
    int dcn3d_backward_input_offset_##SUF(const T* input, const T* weight, const T* offset, const T* grad_output,   \
                                          T* grad_input, T* grad_offset, DCN3D_GEOMETRY, void* workspace,           \
                                          size_t workspace_bytes, void* stream) {                                   \
        return backward_input_offset<T, 3>(geo3(G3_ARGS), input, weight, offset, grad_output, grad_input,           \
                                           grad_offset, workspace, workspace_bytes,                                 \
                                           static_cast<hipStream_t>(stream));                                       \
    }                                                                                                               \
    int dcn3d_backward_input_offset_flags_##SUF(const T* input, const T* weight, const T* offset,                   \
                                                const T* grad_output, T* grad_input, T* grad_offset,                \
                                                DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes,            \
                                                void* stream, unsigned flags) {                                     \
        if (flags & ~(unsigned)DCN_FLAG_OOB_OFFSET_GRAD_ZERO) return fail(DCN_E_ARGUMENT, "unknown flag");          \
        return backward_input_offset<T, 3>(geo3(G3_ARGS), input, weight, offset, grad_output, grad_input,           \
                                           grad_offset, workspace, workspace_bytes,                                 \
                                           static_cast<hipStream_t>(stream), flags);                                \
    }                                                                                                               \
    int dcn3d_backward_weight_##SUF(const T* input, const T* offset, const T* grad_output, T* grad_weight,          \
                                    DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {        \
        return backward_weight<T, 3>(geo3(G3_ARGS), input, offset, grad_output, grad_weight, workspace,             \
                                     workspace_bytes, static_cast<hipStream_t>(stream));                            \
    }                                                                                                               \
    int dcn2d_forward_##SUF(const T* input, const T* weight, const T* offset, const T* bias, T* output,             \
                            DCN2D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {                \
        return forward<T, 2>(geo2(G2_ARGS), input, weight, offset, bias, output, workspace, workspace_bytes,        \
                             static_cast<hipStream_t>(stream));                                                     \
    }                                                                                                               \
    int dcn2d_backward_input_offset_##SUF(const T* input, const T* weight, const T* offset, const T* grad_output,   \
                                          T* grad_input, T* grad_offset, DCN2D_GEOMETRY, void* workspace,           \
                                          size_t workspace_bytes, void* stream) {                                   \
        return backward_input_offset<T, 2>(geo2(G2_ARGS), input, weight, offset, grad_output, grad_input,           \
                                           grad_offset, workspace, workspace_bytes,                                 \
                                           static_cast<hipStream_t>(stream));                                       \
    }                                                                                                               \
    int dcn2d_backward_weight_##SUF(const T* input, const T* offset, const T* grad_output, T* grad_weight,          \
                                    DCN2D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {        \
        return backward_weight<T, 2>(geo2(G2_ARGS), input, offset, grad_output, grad_weight, workspace,             \
                                     workspace_bytes, static_cast<hipStream_t>(stream));                            \
    }

DEFINE_OPS(f32, float)
DEFINE_OPS(f64, double)

size_t conv2d_workspace_bytes(int elem_size, int batch, int input_c, int output_c, size_t input_volume, size_t output_volume,
                              int kernel_volume, int group) {
    const size_t inner = dcn_workspace_bytes_for(elem_size, batch, input_c, output_c, input_volume, output_volume, kernel_volume,
                                                 group, input_c);
    if (!inner || elem_size == 2) return 0;
    const size_t zb = elem_size == 8 ? conv2d_zero_bytes<double>(batch, kernel_volume, output_volume)
                                     : conv2d_zero_bytes<float>(batch, kernel_volume, output_volume);
    return inner + 2 * zb;
}
size_t conv2d_layer_backward_workspace_bytes(int elem_size, int batch, int input_c, int output_c, size_t input_volume, size_t output_volume, int kernel_volume,
                                             int group) {
    size_t data = conv2d_workspace_bytes(elem_size, batch, input_c, output_c, input_volume, output_volume, kernel_volume, group);
    if (!data || input_c % group || output_c % group) return 0;
    if (elem_size == 8) return data + align256(backward_weight_need<double>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group));
    const size_t fwd = forward_need<float>(batch, output_c, input_c, input_volume, kernel_volume, group, output_c);      // grad_output -> grad_input
    return (fwd > data ? fwd : data) + align256(backward_weight_need<float>(batch, input_c, output_c, input_volume, output_volume, kernel_volume, group));
}
#define C2_ARGS batch, input_c, output_c, input_h, input_w, output_h, output_w, kernel_h, kernel_w, pad_h, pad_w, \
                stride_h, stride_w, dilation_h, dilation_w, input_c, group
#define DEFINE_CONV2D(SUF, T)                                                                                       \
    int conv2d_forward_##SUF(const T* input, const T* weight, const T* bias, T* output, CONV2D_GEOMETRY,            \
                             void* workspace, size_t workspace_bytes, void* stream) {                               \
        return conv2d_forward<T>(geo2(C2_ARGS), input, weight, bias, output, workspace, workspace_bytes,            \
                                 static_cast<hipStream_t>(stream));                                                 \
    }                                                                                                               \
    int conv2d_backward_input_##SUF(const T* weight, const T* grad_output, T* grad_input, CONV2D_GEOMETRY,          \
                                    void* workspace, size_t workspace_bytes, void* stream) {                        \
        return conv2d_backward_input<T>(geo2(C2_ARGS), weight, grad_output, grad_input, workspace, workspace_bytes, \
                                        static_cast<hipStream_t>(stream));                                          \
    }                                                                                                               \
    int conv2d_backward_weight_##SUF(const T* input, const T* grad_output, T* grad_weight, CONV2D_GEOMETRY,         \
                                     void* workspace, size_t workspace_bytes, void* stream) {                       \
        return conv2d_backward_weight<T>(geo2(C2_ARGS), input, grad_output, grad_weight, workspace,                 \
                                         workspace_bytes, static_cast<hipStream_t>(stream));                        \
    }
DEFINE_CONV2D(f32, float)
DEFINE_CONV2D(f64, double)
#define DEFINE_CONV2D_LAYER(SUF, T)                                                                                 \
    int conv2d_layer_backward_##SUF(const T* input, const T* weight, const T* grad_output, T* grad_input,           \
                                    T* grad_weight, T* grad_bias, CONV2D_GEOMETRY, void* workspace,                 \
                                    size_t workspace_bytes, void* stream) {                                         \
        return conv2d_layer_backward<T>(geo2(C2_ARGS), input, weight, grad_output, grad_input, grad_weight,         \
                                        grad_bias, workspace, workspace_bytes, static_cast<hipStream_t>(stream));   \
    }
DEFINE_CONV2D_LAYER(f32, float)
DEFINE_CONV2D_LAYER(f64, double)

#define DEFINE_OPS16(SUF, S)                                                                                        \
    int dcn3d_forward_##SUF(const void* input, const void* weight, const void* offset, const void* bias, void* output, \
                            DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {                \
        return forward16<S, 3>(geo3(G3_ARGS), (const S*)input, (const S*)weight, (const S*)offset, (const S*)bias,  \
                               (S*)output, workspace, workspace_bytes, static_cast<hipStream_t>(stream));           \
    }                                                                                                               \
    int dcn3d_backward_input_offset_##SUF(const void* input, const void* weight, const void* offset,                \
                                          const void* grad_output, void* grad_input, void* grad_offset,             \
                                          DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {  \
        return backward_input_offset16<S, 3>(geo3(G3_ARGS), (const S*)input, (const S*)weight, (const S*)offset,    \
                                             (const S*)grad_output, (S*)grad_input, (S*)grad_offset, workspace,     \
                                             workspace_bytes, static_cast<hipStream_t>(stream));                    \
    }                                                                                                               \
    int dcn3d_backward_weight_##SUF(const void* input, const void* offset, const void* grad_output,                 \
                                    void* grad_weight, DCN3D_GEOMETRY, void* workspace, size_t workspace_bytes,     \
                                    void* stream) {                                                                 \
        return backward_weight16<S, 3>(geo3(G3_ARGS), (const S*)input, (const S*)offset, (const S*)grad_output,     \
                                       (S*)grad_weight, workspace, workspace_bytes,                                 \
                                       static_cast<hipStream_t>(stream));                                           \
    }                                                                                                               \
    int dcn2d_forward_##SUF(const void* input, const void* weight, const void* offset, const void* bias, void* output, \
                            DCN2D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {                \
        return forward16<S, 2>(geo2(G2_ARGS), (const S*)input, (const S*)weight, (const S*)offset, (const S*)bias,  \
                               (S*)output, workspace, workspace_bytes, static_cast<hipStream_t>(stream));           \
    }                                                                                                               \
    int dcn2d_backward_input_offset_##SUF(const void* input, const void* weight, const void* offset,                \
                                          const void* grad_output, void* grad_input, void* grad_offset,             \
                                          DCN2D_GEOMETRY, void* workspace, size_t workspace_bytes, void* stream) {  \
        return backward_input_offset16<S, 2>(geo2(G2_ARGS), (const S*)input, (const S*)weight, (const S*)offset,    \
                                             (const S*)grad_output, (S*)grad_input, (S*)grad_offset, workspace,     \
                                             workspace_bytes, static_cast<hipStream_t>(stream));                    \
    }                                                                                                               \
    int dcn2d_backward_weight_##SUF(const void* input, const void* offset, const void* grad_output,                 \
                                    void* grad_weight, DCN2D_GEOMETRY, void* workspace, size_t workspace_bytes,     \
                                    void* stream) {                                                                 \
        return backward_weight16<S, 2>(geo2(G2_ARGS), (const S*)input, (const S*)offset, (const S*)grad_output,     \
                                       (S*)grad_weight, workspace, workspace_bytes,                                 \
                                       static_cast<hipStream_t>(stream));                                           \
    }

DEFINE_OPS16(bf16, Bf16)
DEFINE_OPS16(f16, Fp16)

}  // extern "C"
