// Host side shared by the translation units of libdcn_amd.so: argument validation, workspace layout,
// tuning knobs, halo tiling plans, launch helpers, and the operator functions behind the C ABI.
#pragma once
#include "../../include/dcn_amd.h"
#include "dcn_kernels.h"
#include "dcn_forward.h"
#include "dcn_forward_split.h"
#include "dcn_forward_plain.h"
#include "dcn_prepare.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>
#include <utility>

namespace dcn {

inline thread_local std::string g_err;

inline int fail(int code, const char* msg) {
    g_err = msg;
    return code;
}


// Largest re-laid-out weight any call needs; see relayout_weight_kernel for the two layouts.
template <typename T> inline void fwd_weight_pad(int M, int Cg, int& MT, int& mchunks, int& Mp, int& Cgp) {
    const int TN = Mma<T>::TN, KL = Mma<T>::KL;
    const int mtiles = (M + TN - 1) / TN;
    MT = mtiles >= 8 ? 8 : (mtiles > 2 ? 4 : mtiles);          // 1, 2, 4 or 8 tiles per wavefront
    mchunks = (mtiles + MT - 1) / MT;
    Mp = mchunks * MT * TN;
    Cgp = Cg + 2 * KL;       // the kernels read up to one reduction step past the last channel
}
// backward-data layout.  MK = reduction steps over output channels whose grad_output values
// backward_data_kernel keeps in registers (0: M too large, the kernel re-reads grad_output per tap).
template <typename T> inline int bwd_data_mk(int M) {
    const int steps = (M + Mma<T>::KL - 1) / Mma<T>::KL;
    for (int mk = 8; mk <= 64; mk *= 2)
        if (steps <= mk) return mk;
    return 0;
}
template <typename T> inline void bwd_data_weight_pad(int M, int Cg, int& Mp, int& Cgp) {
    // rows: reduction steps are consumed in batches of 8; the coordinate kernel reads up to KL rows further
    const int KL = Mma<T>::KL;
    const int steps = ((M + KL - 1) / KL + 7) / 8 * 8;
    Mp = steps * KL + KL;
    const int mk = bwd_data_mk<T>(M) * KL;
    if (mk > Mp) Mp = mk;
    Cgp = Cg + Mma<T>::TN;
}
inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

constexpr int TAP_PAD = 8;      // zero tap slabs behind the last group: an MFMA pass may start up to 7 taps before the end
// Elements of the per-chunk weight slabs of the fused backward kernel (pack_backward_weight, chunks of
// `cch` channels) for `slabs` slabs.
template <typename T, typename S = T> inline size_t packed_weight_elems(int M, int kV, size_t slabs, int cch) {
    const int TP = Mma<T>::TN / cch;
    return slabs * ((kV + TP - 1) / TP) * (size_t)gcol_slab_steps<T, S>(M) * 64 * (std::is_same<S, T>::value ? 1 : 4);
}
// Upper bound of chunk_slot<cch>(cpg, Cg, c) + 1 over the channels: the slabs a per-chunk weight
// layout occupies.  cpg = 0: the channels per deformable group are not known (the first workspace
// query is not told them) and the bound assumes their largest possible number of groups, C_in.
inline size_t slab_bound(size_t C_in, int G, int cpg, int cch) { return C_in / cch + (cpg > 0 ? C_in / cpg : C_in) + G + 1; }
// Any weight layout of backward_input_offset fits but that of backward_fused_kernel.
template <typename T> inline size_t bwd_data_weight_bytes(int M, int Cg, int kV, int G, int cpg = 0) {
    int Mp, Cgp;
    bwd_data_weight_pad<T>(M, Cg, Mp, Cgp);
    const size_t plain = ((size_t)G * kV + TAP_PAD) * Mp * Cgp;
    const size_t C_in = (size_t)Cg * G;
    const size_t packed4 = packed_weight_elems<T>(M, kV, slab_bound(C_in, G, cpg, 4), 4);
    const size_t packed8 = packed_weight_elems<T>(M, kV, slab_bound(C_in, G, cpg, 8), 8);
    const size_t packed16 = packed_weight_elems<T>(M, kV, slab_bound(C_in, G, cpg, 16), 16);
    size_t packed = packed4 > packed8 ? packed4 : packed8;
    if (packed16 > packed) packed = packed16;
    return align256((plain > packed ? plain : packed) * sizeof(T));
}
// ... and that one too (float32 and 16-bit storage; float64 has another kernel): S the storage format
template <typename T, typename S = T> inline size_t bwd_fused_weight_bytes(int M, int Cg, int kV, int G, int cpg = 0) {
    size_t bytes = bwd_data_weight_bytes<T>(M, Cg, kV, G, cpg);
    if constexpr (sizeof(T) == 4)
        for (int cch = 4; cch <= 16; cch *= 2) {
            const size_t parts = slab_bound((size_t)Cg * G, G, cpg, cch) * fused_slab_ops<S>(M, kV, cch) * 16;
            if (parts > bytes) bytes = parts;
        }
    return align256(bytes);
}
// Partial outputs of a forward pass that splits the input channels of a position block over several
// workgroups: only layers of few positions do (too few blocks to fill the device), with at most
// FWD_MAX_SPLIT parts and FWD_PARTIAL_CAP bytes.
constexpr int FWD_MAX_SPLIT = 16;
constexpr size_t FWD_PARTIAL_CAP = (size_t)64 << 20;
constexpr size_t FWD_SPLIT_POSITIONS = 256 * 512;      // no split from this many positions on: they fill the device anyway
inline size_t forward_partial_bound(int N, int C_out, size_t outV, size_t elem) {
    if ((size_t)N * outV >= FWD_SPLIT_POSITIONS) return 0;
    const size_t all = (size_t)FWD_MAX_SPLIT * N * C_out * outV * elem;
    return align256(all < FWD_PARTIAL_CAP ? all : FWD_PARTIAL_CAP) + 256;
}
// last bytes of a backward_input_offset workspace: bounds of the weights, and the plan chosen on the device
constexpr size_t BWD_TAIL = BOUND_BLOCKS * 2 * sizeof(float) + 256;
template <typename T> inline size_t forward_need(int N, int C_in, int C_out, size_t outV, int kV, int G, int cpg = 0) {
    const int M = C_out / G, Cg = C_in / G;
    int MT, mchunks, Mp, Cgp;
    fwd_weight_pad<T>(M, Cg, MT, mchunks, Mp, Cgp);
    // [g][tap][c][m] for the kernel without LDS tiling, or one slab per four (float64) or eight
    // channels for the halo kernels (their row padding is at most eight tiles' worth)
    const int TNf = Mma<T>::TN;
    const int Mp8 = ((M + TNf - 1) / TNf + 7) / 8 * 8 * TNf;
    const size_t fwd_plain = (size_t)G * kV * (Mp > Mp8 ? Mp : Mp8) * Cgp * sizeof(T);
    const size_t fwd_quad = sizeof(T) == 4 ? slab_bound((size_t)C_in, G, cpg, FG) * split_slab_elems<float>(kV, Mp8) * 2
                                           : slab_bound((size_t)C_in, G, cpg, FQ) * forward_slab_elems<T>(kV, Mp8) * sizeof(T);
    return (fwd_plain > fwd_quad ? fwd_plain : fwd_quad) + forward_partial_bound(N, C_out, outV, sizeof(T)) + 1024;
}
// The allocation-free entry point accepts a layer by the size of its weight re-laid out as float32 (the larger of
// [g][tap][c][m] and one slab per four channels).  What the halo kernels then store is three bfloat16 parts per
// weight in slabs of eight channels: half as much again, and three times as much where the deformable groups have
// four channels, each of which takes a slab.  The array holds that for every layer accepted (behind it 256 bytes
// that operands of half a group are read past the end, and the block of the plan word).
constexpr size_t NOALLOC_ARRAY_BYTES = 3 * (size_t)DCN_NOALLOC_SCRATCH_BYTES + 4096;
inline size_t noalloc_weight_bytes(const Params& P) {
    int MT, mchunks, Mp, Cgp;
    fwd_weight_pad<float>(P.M, P.Cg, MT, mchunks, Mp, Cgp);
    const int Mp8 = ((P.M + 31) / 32 + 7) / 8 * 8 * 32;
    const size_t plain = (size_t)P.G * P.kV * (Mp > Mp8 ? Mp : Mp8) * Cgp * sizeof(float);
    const size_t quad = ((size_t)chunk_slot<FQ>(P.cpg, P.Cg, P.C_in - 1) + 1) * forward_slab_elems<float>(P.kV, Mp8) * sizeof(float);
    return plain > quad ? plain : quad;
}
// Bytes of the halo kernels' packed weights (float32: three parts, 16-bit storage: one).
template <typename S> inline size_t split_weight_bytes(const Params& P, int Mp) {
    return ((size_t)chunk_slot<FG>(P.cpg, P.Cg, P.C_in - 1) + 1) * split_slab_elems<S>(P.kV, Mp) * 2 + 256;      // (+: operands read from four elements further on)
}
// grad_output in the operand order of backward_fused_kernel (float64: another kernel)
template <typename S> inline size_t fused_gout_need(int N, int M, int G, size_t outV) {
    if constexpr (sizeof(S) == 8) return 0;
    else return align256(fused_gout_bytes<S>(N, M, G, outV));
}
// packed weights, two channels-last tensors, grad_output in operand order (float32 and 16-bit storage), the tail
template <typename T, typename S = T> inline size_t backward_data_need(int N, int C_in, int C_out, size_t inV, size_t outV, int kV, int G, int cpg = 0) {
    return bwd_fused_weight_bytes<T, S>(C_out / G, C_in / G, kV, G, cpg) + 2 * align256((size_t)N * C_in * inV * sizeof(T)) +
           fused_gout_need<S>(N, C_out / G, G, outV) + BWD_TAIL + 512;
}
// Where the parts of a backward_input_offset workspace lie: [ packed weights | input channels-last | its gradient channels-last |
// grad_output in operand order | ... | tail ].  A workspace without room for all of it -- what dcn_workspace_bytes asks for has --
// is laid out for the kernels that use neither the packed parts nor grad_output in operand order (`fused` false), as long as it holds
// the weights of those and the two channels-last regions.
struct DataLayout {
    size_t wbytes, tbytes;      // packed weights; one channels-last region
    size_t gq_at;
    bool fused;
    // Bounds of the weights and, 64 bytes into the block behind them, the plan chosen on the device: in the last whole 256-byte blocks
    // of the workspace where those lie behind the channels-last regions (tail_words), else at the start of the channels-last
    // gradient, which the LDS paths do not use.
    size_t tail_at;
    bool tail_words;
};
template <typename T, typename S> inline int data_layout(const Params& P, size_t ws_bytes, DataLayout& l) {
    l.tbytes = align256((size_t)P.N * P.C_in * P.inV * sizeof(T));
    const size_t tail = ws_bytes >= BWD_TAIL ? (ws_bytes - 256) / 256 * 256 - (BWD_TAIL - 256) : 0;
    for (const bool fused : {true, false}) {
        l.fused = fused;
        l.wbytes = fused ? bwd_fused_weight_bytes<T, S>(P.M, P.Cg, P.kV, P.G, P.cpg) : bwd_data_weight_bytes<T>(P.M, P.Cg, P.kV, P.G, P.cpg);
        l.gq_at = l.wbytes + 2 * l.tbytes;
        l.tail_words = tail >= l.gq_at;
        l.tail_at = l.tail_words ? tail : l.wbytes + l.tbytes;
        if (l.tail_words && ws_bytes >= l.gq_at + fused_gout_need<S>(P.N, P.M, P.G, P.outV) + BWD_TAIL + 256) break;
    }
    if (ws_bytes < l.gq_at || (!l.tail_words && l.tbytes < BWD_TAIL)) return fail(DCN_E_WORKSPACE, "workspace too small");
    return DCN_OK;
}
// A channels-last copy of the input, grad_output channels-last or (float32) in operand order + one partial weight per position split (at most 256 splits, and never more
// than about 4096 workgroups: see bww_plan) + the strips of grad_output's sums
template <typename T> inline size_t backward_weight_need(int N, int C_in, int C_out, size_t inV, size_t outV, int kV, int G) {
    const int TNq = Mma<T>::TN;
    const long long tiles_lb = (long long)kV * ((C_in + TNq - 1) / TNq);           // lower bound of kV * nct * mchunks
    long long split_ub = (4096 + tiles_lb - 1) / tiles_lb;
    if (split_ub > 256) split_ub = 256;
    if (split_ub < 1) split_ub = 1;
    const size_t obytes = (size_t)N * C_out * outV * sizeof(T), rbytes = sizeof(T) == 4 && (kV > 1 || C_out / G > 32) ? row_operand_bytes<float>(N, C_out, outV) : 0;
    return align256((size_t)N * C_in * inV * sizeof(T)) + align256(obytes > rbytes ? obytes : rbytes) +
           align256((size_t)split_ub * kV * C_out * (C_in / G) * sizeof(T)) + align256((size_t)N * last_strips((unsigned)outV) * C_out * sizeof(T));
}
template <typename T> inline size_t workspace_need(int N, int C_in, int C_out, size_t inV, size_t outV, int kV, int G, int cpg = 0) {
    const size_t fwd = forward_need<T>(N, C_in, C_out, outV, kV, G, cpg), bwd = backward_data_need<T>(N, C_in, C_out, inV, outV, kV, G, cpg),
                 bww = backward_weight_need<T>(N, C_in, C_out, inV, outV, kV, G);
    const size_t need = fwd > bwd ? fwd : bwd;
    return need > bww ? need : bww;
}

// The workspace of a layer's backward pass: [ 16-bit storage: float gradients | backward_input_offset | backward_weight ], and in the place
// of the last two, once the kernels that read 16-bit tensors have run, [ float copies of the tensors | an operator on them ] for what
// they decline (the query is not told the strides and dilations that decide it).
struct LayerNeed { size_t grads, data, weight, copies, wide; };
template <typename T, typename S> inline LayerNeed layer_need(int nd, int N, int C_in, int C_out, size_t inV, size_t outV, int kV, int G, int cpg) {
    const size_t in = (size_t)N * C_in * inV, w = (size_t)C_out * (C_in / G) * kV, off = (size_t)N * (C_in / cpg) * kV * nd * outV, out = (size_t)N * C_out * outV;
    LayerNeed n = {};
    n.data = align256(backward_data_need<T, S>(N, C_in, C_out, inV, outV, kV, G, cpg));
    n.weight = align256(backward_weight_need<T>(N, C_in, C_out, inV, outV, kV, G));
    if (!std::is_same<S, T>::value) {
        n.grads = align256(in * sizeof(T)) + align256(off * sizeof(T)) + align256(w * sizeof(T)) + align256((size_t)C_out * sizeof(T));
        n.copies = align256(in * sizeof(T)) + align256(off * sizeof(T)) + align256(w * sizeof(T)) + align256(out * sizeof(T));
        n.wide = align256(backward_data_need<T>(N, C_in, C_out, inV, outV, kV, G, cpg));
        if (n.weight > n.wide) n.wide = n.weight;
    }
    return n;
}
inline size_t layer_bytes(const LayerNeed& n) {
    const size_t native = n.data + n.weight, wide = n.copies + n.wide;
    return n.grads + (native > wide ? native : wide);
}

struct Geometry {   // the reference's argument list, 2-D mapped onto slots 1,2 with a unit length axis
    int nd, N, C_in, C_out, in[3], out[3], k[3], pad[3], stride[3], dil[3], cpg, G;
};

// Mirrors shape_check of the reference as far as it can be stated without tensor handles
// (deform3d/lib/deform_conv3d_cuda.cpp:24-87): the extents must be consistent with each other and
// with the output-size formula.  Rank and per-tensor size checks live in the Python front end,
// which owns the tensors.
inline int validate(const Geometry& g, Params& P) {
    if (g.N <= 0 || g.C_in <= 0 || g.C_out <= 0) return fail(DCN_E_ARGUMENT, "batch / channel extents must be positive");
    if (g.G <= 0 || g.C_in % g.G || g.C_out % g.G) return fail(DCN_E_ARGUMENT, "input c != kernel c");
    if (g.cpg <= 0 || g.C_in % g.cpg) return fail(DCN_E_ARGUMENT, "off channel");
    static const char* const omsg[3] = {"error output ll", "error outhh", "error outww"};
    for (int a = 3 - g.nd; a < 3; ++a) {
        if (g.in[a] <= 0 || g.k[a] <= 0 || g.stride[a] <= 0 || g.dil[a] <= 0 || g.pad[a] < 0)
            return fail(DCN_E_ARGUMENT, "input / kernel / stride / dilation extents must be positive, pad non-negative");
        if (g.in[a] + 2 * g.pad[a] - g.k[a] < 0) return fail(DCN_E_ARGUMENT, omsg[a]);
        // the reference's dilation-blind output size, or the usual dilation-aware one (the sampler
        // gives every position a meaning, so both are served)
        const int blind = (g.in[a] + 2 * g.pad[a] - g.k[a]) / g.stride[a] + 1;
        const int span = g.in[a] + 2 * g.pad[a] - g.dil[a] * (g.k[a] - 1) - 1;
        const int standard = span >= 0 ? span / g.stride[a] + 1 : 0;
        if (g.out[a] != blind && !(standard >= 1 && g.out[a] == standard)) return fail(DCN_E_ARGUMENT, omsg[a]);
    }
    const long long inV = (long long)g.in[0] * g.in[1] * g.in[2], outV = (long long)g.out[0] * g.out[1] * g.out[2];
    // per-channel offsets are 32-bit inside the kernels (including a bias of up to 4 channels)
    if (inV > (1ll << 27) || outV > (1ll << 27)) return fail(DCN_E_ARGUMENT, "a single channel exceeds 2^27 voxels");
    // channels-last voxel*channel offsets of one sample are 32-bit as well
    if (inV * g.C_in > (1ll << 31)) return fail(DCN_E_ARGUMENT, "one input sample exceeds 2^31 elements");
    if (g.N > 65535) return fail(DCN_E_ARGUMENT, "batch exceeds 65535");
    P.oob_zero = P.transposed = 0;
    P.nd = g.nd; P.N = g.N; P.C_in = g.C_in; P.C_out = g.C_out; P.G = g.G; P.cpg = g.cpg; P.DG = g.C_in / g.cpg;
    P.M = g.C_out / g.G; P.Cg = g.C_in / g.G;
    for (int a = 0; a < 3; ++a) {
        P.in[a] = g.in[a]; P.out[a] = g.out[a]; P.k[a] = g.k[a];
        P.pad[a] = g.pad[a]; P.stride[a] = g.stride[a]; P.dil[a] = g.dil[a];
    }
    P.inV = (unsigned)inV; P.outV = (unsigned)outV; P.kV = g.k[0] * g.k[1] * g.k[2];
    P.tiles = P.mchunks = P.Mp = P.Cgp = P.nsplit = P.nctiles = 0;
    return DCN_OK;
}

inline int check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_err = std::string(what) + ": " + hipGetErrorString(e);
        return DCN_E_LAUNCH;
    }
    return DCN_OK;
}

template <typename T>
inline int relayout(const Params& P, const T* w, T* wt, int channel_fastest, hipStream_t s) {
    const size_t total = (size_t)P.G * P.kV * P.Mp * P.Cgp;
    const int blocks = (int)((total + 255) / 256 > 4096 ? 4096 : (total + 255) / 256);
    hipLaunchKernelGGL(relayout_weight_kernel<T>, dim3(blocks), dim3(256), 0, s, P, w, wt, channel_fastest);
    return check_launch("relayout_weight_kernel");
}

// ---------------------------------------------------------------------------------------------
// Halo tiling plan: block of output positions per workgroup, halo extents, channels per LDS pass.
// Returns false when the geometry does not suit (halo too large for the staging table or LDS).
// Tuning knobs (environment, read once per process):
//   DCN_HALO_MARGIN        voxels of halo beyond the integer tap span on each side: one fixed margin instead of
//                          the choice on the device among 2, 3, 4 (3-D) or 2, 4, 6 (2-D)
//   DCN_ADAPTIVE_MARGIN=0  always the smallest of those margins (2)
//   DCN_TRACE_PLANS=1      print the halo plans and launches of every call on stderr
//   DCN_LDS_BUDGET_KB      LDS per 512-thread workgroup of the forward halo kernel (default 72: two per CU)
//   DCN_FORWARD_WG=512     never use the 1024-thread forward variant; =1024 use it whenever its halo fits
//   DCN_FORWARD_SPLIT=n    forward pass, float32 and float64: split the input channels of a position block over at most n workgroups (0: never)
//   DCN_FORWARD_TAIL=0     forward pass: never split only the units of the last, partly filled round of workgroups (n > 1: n ways)
//   DCN_FORWARD_TAIL2=0    forward pass: the split units of the last round all the same number of ways, never in two runs
//   DCN_FORWARD_SLOTS=n    forward pass: plan the launch as if n workgroups ran at once (test hook)
//   DCN_FORWARD_SHARED=0   forward pass, float32 and 16-bit: never share the sampled columns of a block among wavefronts
//   DCN_FORWARD_SMALL=0    forward pass, float32 and 16-bit: never several wavefronts to a position
//   DCN_FORWARD_TINY=0     ... never more than four; 1 / 2 (test hook): sixteen to blocks of 32 positions / eight to blocks of 64 on every
//                          layer with several, of up to two row tiles
//   DCN_PLAIN=0            the plain convolution of float32 on the kernels of the deformable layer; =2 (test hook): of any size on its own
//   DCN_SCATTER_BUDGET_KB  dynamic LDS per workgroup of the privatised scatter kernels (default 156, at most 157: backward_fused_kernel, 144, at
//                          most 159: the others)
//   DCN_SCATTER=global     scatter grad-input with global atomics instead of the LDS-privatised kernel
//   DCN_COORD=separate     grad_offset from the channels-last kernel instead of the fused LDS-halo kernel
// Both kernels that form grad_input and grad_offset over a halo, backward_fused_kernel and backward_input_halo_kernel:
//   DCN_FUSED_WAVES=4      blocks of 128 positions in the shape with the smallest halo even where 256 fit (the second: four wavefronts)
//   DCN_FUSED_CHUNK=4      4-channel chunks also where they would take 8 or 16; =8: never 16 (2-D layers)
//   DCN_FUSED_TAIL=0       all items split alike, never only those of the last round
//   DCN_CSPLIT=n           every item split over n workgroups
//   DCN_FUSED_SLOTS=n      plan the launch as if n workgroups ran at once (test hook)
//   DCN_FUSED_PAIR=0       float32: one channel per 64-bit LDS cell instead of two 32-bit halves, and never backward_fused_kernel
// backward_input_halo_kernel alone:
//   DCN_FUSED_FIXED=0      runtime plane stride even where the compile-time one fits
//   DCN_FUSED_BREG2=0      no second register set for the grad_output operand of 64 < M <= 128
//   DCN_GLOBAL_PLAN=0      backward_input_offset (3-D): the device is not offered the path without LDS tiling
//   DCN_NATIVE16=0         16-bit entry points: always widen to float32 and run the float32 kernels
static size_t env_kb(const char* name, int dflt) {
    const char* e = getenv(name);
    const int v = e ? atoi(e) : dflt;
    return (size_t)(v > 0 ? v : dflt) * 1024;
}
static size_t lds_budget() { static const size_t v = env_kb("DCN_LDS_BUDGET_KB", 72); return v; }
// (at most what a CU has beside what the kernels declare themselves: backward_input_halo_kernel 100 bytes, backward_fused_kernel 2120)
static size_t scatter_budget() { static const size_t v = std::min<size_t>(env_kb("DCN_SCATTER_BUDGET_KB", 144), 159 * 1024); return v; }
static size_t fused_budget() { static const size_t v = std::min<size_t>(env_kb("DCN_SCATTER_BUDGET_KB", 156), 157 * 1024); return v; }
static bool fused_coord() {
    static const int v = [] { const char* e = getenv("DCN_COORD"); return (e && strcmp(e, "separate") == 0) ? 0 : 1; }();
    return v != 0;
}
// What the library needs to know about a GPU, looked up once per device ordinal.
struct DeviceInfo { int state = 0; int cus = 256; };      // state: 0 not looked up, 1 usable, -1 not a gfx950
constexpr int MAX_DEVICES = 64;
inline std::mutex g_device_lock;
inline DeviceInfo g_device[MAX_DEVICES];

// Fills `out` for the current device; DCN_E_DEVICE when there is none or it is not a gfx950.
inline int device_info(const DeviceInfo** out, int* ordinal = nullptr) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        (void)hipGetLastError();
        return fail(DCN_E_DEVICE, "no current HIP device (or its ordinal is beyond 63)");
    }
    std::lock_guard<std::mutex> lock(g_device_lock);
    DeviceInfo& d = g_device[dev];
    if (d.state == 0) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) {
            (void)hipGetLastError();
            return fail(DCN_E_DEVICE, "hipGetDeviceProperties failed");
        }
        d.state = strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : -1;
        if (prop.multiProcessorCount > 0) d.cus = prop.multiProcessorCount;
    }
    if (d.state < 0) return fail(DCN_E_DEVICE, "the current device is not a gfx950 GPU");
    if (out) *out = &d;
    if (ordinal) *ordinal = dev;
    return DCN_OK;
}
static int cu_count() {      // of the current device (every entry point has called device_info by then)
    const DeviceInfo* d = nullptr;
    return device_info(&d) == DCN_OK ? d->cus : 256;
}
static int wide_forward() {      // 0 never, 1 when it pays, 2 whenever the halo fits
    static const int v = [] {
        const char* e = getenv("DCN_FORWARD_WG");
        return !e ? 1 : atoi(e) == 512 ? 0 : atoi(e) == 1024 ? 2 : 1;
    }();
    return v;
}
static bool fused_chunk16() {     // DCN_FUSED_CHUNK=8 (or 4): never take 16-channel chunks in the fused backward kernel
    static const int v = [] { const char* e = getenv("DCN_FUSED_CHUNK"); return (e && (atoi(e) == 8 || atoi(e) == 4)) ? 0 : 1; }();
    return v != 0;
}
static bool fused_chunk8() {      // DCN_FUSED_CHUNK=4: never take 8-channel chunks in the fused backward kernel
    static const int v = [] { const char* e = getenv("DCN_FUSED_CHUNK"); return (e && atoi(e) == 4) ? 0 : 1; }();
    return v != 0;
}
static int fused_first_waves() {
    static const int v = [] { const char* e = getenv("DCN_FUSED_WAVES"); return (e && atoi(e) == 4) ? 4 : 8; }();
    return v;
}
static bool fused_fixed_stride() {      // DCN_FUSED_FIXED=0: runtime plane stride even where the compile-time one fits
    static const int v = [] { const char* e = getenv("DCN_FUSED_FIXED"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool fused_tail_split() {        // DCN_FUSED_TAIL=0: the fused backward kernel never splits only the items of the last round
    static const int v = [] { const char* e = getenv("DCN_FUSED_TAIL"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static int forced_slots() {             // DCN_FUSED_SLOTS=n (test hook): plan the fused backward launch as if n workgroups ran at once
    static const int v = [] { const char* e = getenv("DCN_FUSED_SLOTS"); return e && atoi(e) > 0 ? atoi(e) : 0; }();
    return v;
}
static int forward_split() {            // DCN_FORWARD_SPLIT=n: the forward pass splits the input channels of a position block at most n ways
    static const int v = [] { const char* e = getenv("DCN_FORWARD_SPLIT"); return e ? atoi(e) : 1 << 20; }();
    return v;
}
static int forward_slots() {            // DCN_FORWARD_SLOTS=n (test hook): plan the forward launch as if n workgroups ran at once
    static const int v = [] { const char* e = getenv("DCN_FORWARD_SLOTS"); return e && atoi(e) > 0 ? atoi(e) : 0; }();
    return v;
}
static int forward_tail_split() {       // DCN_FORWARD_TAIL=0: the forward pass never splits the units of its last round of workgroups; n > 1: n ways
    static const int v = [] { const char* e = getenv("DCN_FORWARD_TAIL"); return e ? atoi(e) : 1; }();
    return v;
}
static bool forward_tail_two_runs() {    // DCN_FORWARD_TAIL2=0: the split units of the forward pass's last round are all split the same number of ways
    static const int v = [] { const char* e = getenv("DCN_FORWARD_TAIL2"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static int plain_conv() {                // DCN_PLAIN=0, 2: see above
    static const int v = [] { const char* e = getenv("DCN_PLAIN"); return e ? atoi(e) : 1; }();
    return v;
}
static bool forward_shared() {           // DCN_FORWARD_SHARED=0: the forward pass always samples in every wavefront (forward_split_kernel)
    static const int v = [] { const char* e = getenv("DCN_FORWARD_SHARED"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool forward_small() {            // DCN_FORWARD_SMALL=0: the forward pass never lets several wavefronts share a position
    static const int v = [] { const char* e = getenv("DCN_FORWARD_SMALL"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static int forward_tiny() {              // DCN_FORWARD_TINY=0: at most four wavefronts to a position; 1, 2: see above; -1: unset
    static const int v = [] { const char* e = getenv("DCN_FORWARD_TINY"); return e ? atoi(e) : -1; }();
    return v;
}
static bool fused_pair() {              // DCN_FUSED_PAIR=0: float32 LDS cells of the fused backward kernel hold one channel each (64-bit)
    static const int v = [] { const char* e = getenv("DCN_FUSED_PAIR"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool fused_breg2() {             // DCN_FUSED_BREG2=0: grad_output operand in registers only up to 32 reduction steps
    static const int v = [] { const char* e = getenv("DCN_FUSED_BREG2"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool native16() {                // DCN_NATIVE16=0: the 16-bit entry points always widen to float32 first
    static const int v = [] { const char* e = getenv("DCN_NATIVE16"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool global_plan() {             // DCN_GLOBAL_PLAN=0: the device never chooses the path without LDS tiling
    static const int v = [] { const char* e = getenv("DCN_GLOBAL_PLAN"); return (e && atoi(e) == 0) ? 0 : 1; }();
    return v != 0;
}
static bool scatter_in_lds() {
    static const int v = [] { const char* e = getenv("DCN_SCATTER"); return (e && strcmp(e, "global") == 0) ? 0 : 1; }();
    return v != 0;
}
#define LDS_BUDGET lds_budget()
static int halo_margin() {      // DCN_HALO_MARGIN: one fixed margin; -1 when not set
    static const int v = [] {
        const char* e = getenv("DCN_HALO_MARGIN");
        if (!e) return -1;
        const int m = atoi(e);
        return m < 0 ? 0 : m;
    }();
    return v;
}
// Halo margins to plan for, ascending; the first is the one taken when nothing can be chosen.
static int plan_margins(int nd, int* m) {
    static const int adaptive = [] { const char* e = getenv("DCN_ADAPTIVE_MARGIN"); return (e && atoi(e) == 0) ? 0 : 1; }();
    if (halo_margin() >= 0) { m[0] = halo_margin(); return 1; }
    m[0] = 2;
    if (!adaptive) return 1;
    m[1] = nd == 3 ? 3 : 4;
    m[2] = nd == 3 ? 4 : 6;
    return MAX_PLANS;
}
static_assert(MAX_PLANS == 3, "plan_margins fills three margins");
static bool trace_plans() {             // DCN_TRACE_PLANS=1: the halo plans and launches of every call on stderr
    static const int v = [] { const char* e = getenv("DCN_TRACE_PLANS"); return (e && atoi(e) != 0) ? 1 : 0; }();
    return v != 0;
}
static int default_margin() { return halo_margin() >= 0 ? halo_margin() : 2; }
static int forced_csplit() {    // DCN_CSPLIT=n: workgroups per (tile, deformable group) of the fused backward kernel
    static const int v = [] { const char* e = getenv("DCN_CSPLIT"); return e && atoi(e) > 0 ? atoi(e) : 0; }();
    return v;
}

template <typename T, int ND>
inline bool plan_halo(Params& P, size_t budget, int m, int max_chunk = 1 << 30, size_t cell_bytes = sizeof(T), int waves = WAVESH,
               bool smallest_halo = false, int chunk_mult = 0, const Div* blocks = nullptr, int wmult = 1, bool table = true) {
    const int npos = waves * Mma<T>::TN;        // positions per workgroup, one column tile per wavefront
    int td[3] = {1, 1, 1};
    if (ND == 3) { td[1] = td[2] = npos >= 64 ? 8 : 4; td[0] = npos / (td[1] * td[2]); }
    else         { td[2] = npos >= 128 ? 16 : 8; td[1] = npos / td[2]; }
    if (blocks) {                               // the block shape of another plan
        for (int a = 0; a < 3; ++a) td[a] = blocks[a];
    } else if (smallest_halo) {
        // the block shape (powers of two, at least 4 positions along the fastest axis) with the
        // smallest halo: strided geometries want blocks that are short along the strided axes
        long long best = -1;
        for (int a = 1; a <= npos; a *= 2)
            for (int b = 1; a * b <= npos; b *= 2) {
                const int c = npos / (a * b);
                if (c < 4 || (ND == 2 && a != 1)) continue;
                const int cand[3] = {a, b, c};
                long long hv = 1;
                for (int x = 3 - ND; x < 3; ++x) hv *= (cand[x] - 1) * P.stride[x] + (P.k[x] - 1) * P.dil[x] + 1 + 2 * m;
                if (best < 0 || hv < best) { best = hv; td[0] = a; td[1] = b; td[2] = c; }
            }
    }
    long long hvol = 1, tiles = 1;
    for (int a = 0; a < 3; ++a) {
        P.tdim[a] = td[a];
        P.ntile[a] = (P.out[a] + td[a] - 1) / td[a];
        const bool used = a >= 3 - ND;
        P.mlo[a] = used ? m : 0;
        // lowest corner: base - m; highest corner: base + m (the high corner of a sample at base + m - eps)
        P.hext[a] = used ? (td[a] - 1) * P.stride[a] + (P.k[a] - 1) * P.dil[a] + 1 + 2 * m : 1;
        // (wmult: the innermost extent rounded up to a multiple, for kernels whose LDS layout depends on
        // the position of a halo voxel modulo that number; the extra cells lie on the high side)
        if (a == 2 && wmult > 1) P.hext[a] = (P.hext[a] + wmult - 1) / wmult * wmult;
        hvol *= P.hext[a];
        tiles *= P.ntile[a];
    }
    if (hvol > MAX_HVOL) return false;
    P.hvol = (int)hvol;
    // (table: the kernel keeps an offset per halo voxel in LDS and channel planes of its own stride)
    P.hstride = table ? ((int)hvol + 63) / 64 * 64 + 32 : (int)hvol;
    const size_t tbytes = table ? (size_t)hvol * 4 : 0;
    const int KL = chunk_mult > 0 ? chunk_mult : Mma<T>::KL;      // channels per pass come in multiples of this
    if (budget <= tbytes) return false;
    long long cc = (long long)((budget - tbytes) / ((size_t)P.hstride * cell_bytes));
    cc = cc / KL * KL;
    const int seg = P.cpg < P.Cg ? P.cpg : P.Cg;          // longest run of channels sharing offsets and group
    const int seg_up = (seg + KL - 1) / KL * KL;
    if (cc > seg_up) cc = seg_up;
    if (cc > max_chunk) cc = max_chunk / KL * KL;
    if (cc < KL) return false;
    P.cchunk = (int)cc;
    if (tiles * P.N > 0x7fffffffLL) return false;
    P.tiles = (int)tiles;
    return true;
}

// Raises a kernel's dynamic LDS limit; the runtime is asked only when a kernel needs more than it
// was last granted on the current device.
inline int raise_lds_limit(const void* kern, size_t lds) {
    static std::mutex lock;
    static std::map<std::pair<int, const void*>, size_t> granted;
    int dev = 0;
    if (device_info(nullptr, &dev) != DCN_OK) return DCN_E_DEVICE;
    std::lock_guard<std::mutex> guard(lock);
    size_t& have = granted[std::make_pair(dev, kern)];
    if (lds <= have) return DCN_OK;
    if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        (void)hipGetLastError();
        return fail(DCN_E_LAUNCH, "cannot raise the dynamic LDS limit");
    }
    have = lds;
    return DCN_OK;
}

// Workgroups of a kernel that the current device holds at once (one per CU if the query fails).
inline long long resident_workgroups(const void* kern, int threads, size_t lds) {
    static std::mutex lock;
    static std::map<std::pair<const void*, size_t>, int> per_cu_of;
    int per_cu = 0;
    {
        std::lock_guard<std::mutex> guard(lock);
        int& v = per_cu_of[std::make_pair(kern, lds)];
        if (v == 0) {
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, kern, threads, lds) != hipSuccess || v < 1) {
                (void)hipGetLastError();
                v = 1;
            }
        }
        per_cu = v;
    }
    return (long long)per_cu * cu_count();
}

static HaloPlan halo_plan_of(const Params& P) {
    HaloPlan h;
    for (int a = 0; a < 3; ++a) { h.hext[a] = P.hext[a]; h.mlo[a] = P.mlo[a]; }
    h.hvol = P.hvol; h.hstride = P.hstride; h.cchunk = P.cchunk;
    return h;
}
static bool same_blocks(const Params& a, const Params& b) {
    for (int x = 0; x < 3; ++x)
        if (a.tdim[x] != b.tdim[x] || a.ntile[x] != b.ntile[x]) return false;
    return a.tiles == b.tiles;
}

template <typename K, typename... Args>
inline int launch_halo(K kern, const char* name, dim3 grid, int threads, size_t lds, hipStream_t s, Args... args) {
    if (lds > 48 * 1024)
        if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds)) return rc;
    hipLaunchKernelGGL(kern, grid, dim3(threads), lds, s, args...);
    return check_launch(name);
}

// ---------------------------------------------------------------------------------------------
// The operators, each instantiated in a translation unit of its own (they compile in parallel).
constexpr unsigned FLAG_INPUT_ONLY = 0x100u;     // internal: see backward_input_offset
// off = null (float32): every offset is zero.  transposed: the weight of the convolution that this call is
// the backward pass of.
template <typename T, int ND, typename S = T>
int forward(const Geometry& g, const S* in, const S* w, const S* off, const S* bias, S* out, void* ws, size_t ws_bytes,
            hipStream_t s, bool* declined = nullptr, bool transposed = false);
// prep: jobs that belong to the caller, done in the launch that prepares this operator
template <typename T, int ND, typename S = T>
int backward_input_offset(const Geometry& g, const S* in, const S* w, const S* off, const S* gout, T* gin, T* goff, void* ws,
                          size_t ws_bytes, hipStream_t s, unsigned flags = 0, bool* declined = nullptr, Prep* prep = nullptr);
// backward_weight in two halves: where its operands go (jobs for the preparing launch), and the kernels.
// T arithmetic, S storage (T, or 16 bits: channel pairs, see backward_weight16_kernel).
template <typename T, typename S> struct WeightCall {
    Params P;
    int MT;
    S *in_cl, *gout_cl;
    const S* gout;
    T *partial, *sums;
    int nsums;
    int LW, igroups;                  // > 0: backward_weight_split_kernel, and gout_cl is grad_output in its operand order
};
template <typename T, int ND, typename S>
int backward_weight_plan(const Params& P, const S* in, const S* off, const S* gout, void* ws, size_t ws_bytes, bool bias, WeightCall<T, S>& c, Prep& prep, bool* declined);
template <typename T, int ND, typename S>
int backward_weight_run(const WeightCall<T, S>& c, const S* off, T* gw, T* gb, bool accumulate, hipStream_t s);

template <typename T, typename S>
inline int launch_prepare(const Params& P, const PlanChoice& pc, const Prep& prep, const S* w, const S* off, size_t n_off, hipStream_t s) {
    if (prep.full) return fail(DCN_E_LAUNCH, "too many jobs for the preparing launch");
    if (prep.jobs.n == 0) return DCN_OK;
    hipLaunchKernelGGL((backward_prepare_kernel<T, S>), dim3(prep.blocks), dim3(256), 0, s, P, pc, prep.jobs, w, off, n_off);
    return check_launch("backward_prepare_kernel");
}

}  // namespace dcn
