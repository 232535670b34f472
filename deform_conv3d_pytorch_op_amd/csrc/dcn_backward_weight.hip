// Backward pass to the weight: plans and launches.
#include "dcn_host.h"
#include <cmath>

namespace dcn {

// Plan of backward_weight: channel tiles, m chunks and the number of position splits.
template <typename T>
void bww_plan(const Params& Pin, int& MT, int& mchunks, int& nct, int& nsplit, long long resident = 0) {
    const int TN = Mma<T>::TN;
    const int mtiles = (Pin.M + TN - 1) / TN;
    MT = mtiles > 2 ? 4 : mtiles;
    mchunks = (mtiles + MT - 1) / MT;
    // channel tiles: one per TN channels of every (convolution group x deformable group) segment
    nct = 0;
    for (int gg = 0; gg < Pin.G; ++gg) {
        const int cg0 = gg * Pin.Cg, cg1 = cg0 + Pin.Cg;
        for (int dg = cg0 / Pin.cpg; dg <= (cg1 - 1) / Pin.cpg; ++dg) {
            const int cb = cg0 > dg * Pin.cpg ? cg0 : dg * Pin.cpg;
            const int ce = cg1 < (dg + 1) * Pin.cpg ? cg1 : (dg + 1) * Pin.cpg;
            nct += (ce - cb + TN - 1) / TN;
        }
    }
    // split the position reduction so that the grid holds a few thousand workgroups: the largest
    // whole number of rounds of resident workgroups below about 2560 (a grid just past a whole
    // number of rounds pays a full round for the remainder; more splits mean more partial tiles to
    // write and add up: 4096 measured 1 to 7 % slower on the five benchmark layers)
    constexpr long long BWW_TARGET = 2560;
    const long long slabs = (long long)Pin.N * ((Pin.outV + TN - 1) / TN);
    const long long other = (long long)Pin.kV * nct * mchunks;
    long long split = (BWW_TARGET + other - 1) / other;
    if (resident > 0 && resident <= BWW_TARGET) {
        const long long balanced = (BWW_TARGET / resident) * resident / other;
        if (balanced >= 1 && balanced < split) split = balanced;
    }
    const long long max_split = (slabs + WAVES - 1) / WAVES;
    if (split > max_split) split = max_split;
    if (split > 256) split = 256;
    if (split < 1) split = 1;
    nsplit = (int)split;
}

// Channel tiles of TC channels of the convolution group that has the most, times groups of TP taps.
inline int split_items(const Params& P, int TC, int TP) {
    int most = 0;
    for (int g = 0; g < P.G; ++g) {
        int n = 0;
        for (int dg = g * P.Cg / P.cpg; dg <= ((g + 1) * P.Cg - 1) / P.cpg; ++dg) {
            const int cb = g * P.Cg > dg * P.cpg ? g * P.Cg : dg * P.cpg, ce = (g + 1) * P.Cg < (dg + 1) * P.cpg ? (g + 1) * P.Cg : (dg + 1) * P.cpg;
            n += (ce - cb + TC - 1) / TC;
        }
        most = n > most ? n : most;
    }
    return most * ((P.kV + TP - 1) / TP);
}
// backward_weight_split_kernel takes layers of more than 32 output channels to a group, with items for the four wavefronts of a
// workgroup (not a single tap of few channels) and work for the device: 2.5 slabs to a resident wavefront.  Below, the longer
// preparation and the fuller grid that backward_weight_kernel makes of few items decide (us of a training step, that kernel against
// this one: 45 -> 75 channels, one tap, 15 000 positions 699 : 774; 32 -> 432, 5x5, 612 positions 259 : 265; 32 -> 80, 3x3x3, 1176 positions
// 177 : 184; 96 -> 128, 3x3, 7296 positions 157 : 162); above, this one wins (32 -> 113, 3x3x3, 3456 positions 202 : 183; 16 -> 80, 16 000
// positions 228 : 203; 12 -> 57, 62 000 positions 750 : 698).  Its wavefronts write a partial tile each: about one round of resident
// workgroups, as long as the tiles (written and read at about 8 TB/s) cost less than the longer runs of slabs.
template <typename S> using RowOps = typename Parts<S>::Vec;
template <typename S> using SplitFn = void (*)(Params, const S*, const S*, const S*, const RowOps<S>*, float*, unsigned);
template <int ND, typename S, bool QUAD>
SplitFn<S> split_kernel_of(int MT, int LW, bool plain) {
    if constexpr (ND == 2 && sizeof(S) == 4)
        if (plain) return MT == 4 ? backward_weight_split_kernel<ND, 4, 32, S, QUAD, true> : backward_weight_split_kernel<ND, 2, 32, S, QUAD, true>;
    if constexpr (sizeof(S) == 4)
        if (MT == 8) return backward_weight_split_kernel<ND, 8, 32, S, QUAD>;
    constexpr bool QUAD8 = QUAD && !(ND == 3 && std::is_same<S, Bf16>::value);      // (see split_quad)
    switch (MT * 100 + LW) {
        case 108: return backward_weight_split_kernel<ND, 1, 8, S, QUAD>;
        case 116: return backward_weight_split_kernel<ND, 1, 16, S, QUAD>;
        case 208: return backward_weight_split_kernel<ND, 2, 8, S, QUAD8>;
        case 216: return backward_weight_split_kernel<ND, 2, 16, S, QUAD>;
        case 232: return backward_weight_split_kernel<ND, 2, 32, S, QUAD>;
        case 408: return backward_weight_split_kernel<ND, 4, 8, S, QUAD8>;
        case 416: return backward_weight_split_kernel<ND, 4, 16, S, QUAD>;
        default: return backward_weight_split_kernel<ND, 4, 32, S, QUAD>;
    }
}
template <int ND, typename S>
SplitFn<S> split_kernel(const Params& P, int MT, int LW, bool plain) {
    if constexpr (ND == 3 && sizeof(S) == 4) return split_kernel_of<ND, S, false>(MT, LW, plain);
    else return split_quad<ND, S>(P, MT, LW) ? split_kernel_of<ND, S, true>(MT, LW, plain) : split_kernel_of<ND, S, false>(MT, LW, plain);
}
// Lanes to a tap: 16 or 8 where a segment fits them and that makes fewer items, at 1.05 and 1.2 items for one of 32: eight lanes read 32
// bytes of a corner.  (Longer segments read their cache lines in parts then: 80 -> 96, 3-D, 23 600 positions 406 us a step with 32, 431 with 16.)  Layers of up to 32 output channels, too, if it takes a third off them; the
// first threshold counts items of 32 lanes.  50 training layers, us per step, 32 lanes (or the other
// kernels) : this: 1.058 times as fast on average, at worst 0.994; 16 -> 38 in groups of 4, 3-D, two samples of 16 700 positions in bfloat16 464 : 322; 20 -> 339 in
// groups of 5, 7200 positions 301 : 245; 16 -> 14, 165 000 positions in bfloat16 734 : 602; 24 -> 36 in groups of 6, 10 600 positions 184 : 162.
struct SplitPlan { int MT, LW, mchunks, igroups, nsplit; };     // nsplit 0: not a layer for it, or no room
template <int ND, typename S>
SplitPlan split_plan(const Params& P, bool off, size_t room) {
    SplitPlan c = {};
    const int whole = split_items(P, 32 * lane_channels<S>(), 1);
    int items = whole;
    double least = whole;
    c.LW = 32;
    const int longest = P.cpg < P.Cg ? P.cpg : P.Cg;
    for (int lw : {16, 8}) {
        if (longest > lw * lane_channels<S>()) continue;
        const int n = split_items(P, lw * lane_channels<S>(), 32 / lw);
        const double cost = n * (lw == 8 ? 1.2 : 1.05);
        if (cost >= least || !off) continue;
        least = cost;
        items = n;
        c.LW = lw;
    }
    c.MT = P.M > 64 ? 4 : P.M > 32 ? 2 : 1;
    c.mchunks = ((P.M + 31) / 32 + c.MT - 1) / c.MT;
    c.igroups = (items + WAVES - 1) / WAVES;
    if ((P.M <= 32 && least > 0.67 * whole) || items < WAVES) return c;
    auto resident = [&](int MT) { return (double)resident_workgroups(reinterpret_cast<const void*>(split_kernel<ND, S>(P, MT, c.LW, false)), WG, 0); };
    const long long nslabs = (long long)P.N * (row_steps(P.outV) / 2);
    const double fit = resident(c.MT), other = (double)c.igroups * P.G;
    if ((double)whole * c.mchunks * P.G * (double)nslabs < 2.5 * WAVES * fit) return c;
    const size_t one = (size_t)P.kV * P.C_out * P.Cg * sizeof(float);
    const long long most = (long long)(room / one);
    SplitCost best = split_cost(other * c.mchunks, fit, nslabs, most, one);
    // Eight row tiles in float32, where they hold no more padding than fours do and leave work for the wavefronts that then fit, if that is faster by the estimate.
    const int mtiles = (P.M + 31) / 32, fewer = (mtiles + 7) / 8;
    if (sizeof(S) == 4 && off && c.LW == 32 && fewer * 8 == c.mchunks * 4) {
        const double fit8 = resident(8);
        if ((double)whole * fewer * P.G * (double)nslabs >= 2.5 * WAVES * fit8) {
            const SplitCost eight = split_cost(other * fewer, fit8, nslabs, most, one);
            if (eight_tiles_pay(ND, best, eight)) {
                best = eight;
                c.MT = 8;
                c.mchunks = fewer;
            }
        }
    }
    c.nsplit = best.nsplit;
    if (other * c.mchunks * c.nsplit > 2147483647.0) c.nsplit = 0;
    return c;
}

// Workgroups of backward_weight_kernel that the device holds at once (0 if the query fails).
template <typename T, int ND, int MT>
long long bww_resident() {
    static const long long v = [] {
        int per_cu = 0;
        const size_t lds = (size_t)WAVES * Mma<T>::TN * (Mma<T>::TN + 1) * sizeof(T);
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, backward_weight_kernel<T, ND, MT>, WG, lds) != hipSuccess) {
            (void)hipGetLastError();
            return 0LL;
        }
        return (long long)per_cu * cu_count();
    }();
    return v;
}

template <typename T, int ND, int MT>
int launch_bwd_weight(const WeightCall<T, T>& c, const T* off, hipStream_t s) {
    const Params& P = c.P;
    const int TN = Mma<T>::TN;
    const size_t lds = (size_t)WAVES * TN * (TN + 1) * sizeof(T);
    auto kern = backward_weight_kernel<T, ND, MT>;
    if constexpr (ND == 2)
        if (!off) kern = backward_weight_kernel<T, ND, MT, true>;
    if (lds > 48 * 1024)
        if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds)) return rc;
    const dim3 grid((unsigned)P.nsplit * P.kV * P.nctiles * P.mchunks);
    hipLaunchKernelGGL(kern, grid, dim3(WG), lds, s, P, (const T*)c.in_cl, off, (const T*)c.gout_cl, c.partial);
    return check_launch("backward_weight_kernel");
}

// Workspace of backward_weight: [ input channels-last | grad_output channels-last | partial tiles per
// split | strips of grad_output's sums (bias) ].  S = T: any layer.  16-bit storage: channels-last copies
// in their storage format; declined (nothing planned) where the kernel's 4-byte loads of channel pairs
// would not be aligned (an odd number of input channels, or segments -- intersections of convolution groups
// and deformable groups -- that start at odd channels), where the float32 kernel is the faster one, or
// where the workspace is too small.
template <typename T, int ND, typename S>
int backward_weight_plan(const Params& Pin, const S* in, const S* off, const S* gout, void* ws, size_t ws_bytes, bool bias, WeightCall<T, S>& c, Prep& prep, bool* declined) {
    constexpr bool S16 = !std::is_same<S, T>::value;
    Params& P = c.P;
    P = Pin;
    if (declined) *declined = S16;
    auto refuse = [&](int code, const char* msg) { return S16 ? DCN_OK : fail(code, msg); };
    if ((long long)P.outV * P.C_out > (1ll << 31)) return refuse(DCN_E_ARGUMENT, "one output sample exceeds 2^31 elements");
    if (2 * (long long)P.N > 65535) return refuse(DCN_E_ARGUMENT, "backward_weight: batch exceeds 32767");
    // the kernel addresses both operands by 32-bit byte offsets from the sample's base
    if ((unsigned long long)P.inV * P.C_in * sizeof(S) >= (1ull << 32) || (unsigned long long)P.outV * P.C_out * sizeof(S) >= (1ull << 32))
        return refuse(DCN_E_ARGUMENT, "one sample of the input or of grad_output reaches 4 GiB");
    if constexpr (!S16) {
        int mchunks;
        bww_plan<T>(P, c.MT, mchunks, P.nctiles, P.nsplit);
        const long long resident = c.MT == 1 ? bww_resident<T, ND, 1>() : c.MT == 2 ? bww_resident<T, ND, 2>() : bww_resident<T, ND, 4>();
        bww_plan<T>(P, c.MT, mchunks, P.nctiles, P.nsplit, resident);
        P.mchunks = mchunks;
        if ((long long)P.nsplit * P.kV * P.nctiles * P.mchunks > 0x7fffffffLL) return fail(DCN_E_ARGUMENT, "too many workgroups for one launch");
    } else {
        const int TN = Mma<float>::TN, CT = 2 * TN;
        if (P.C_in % 2 || P.cpg % 2 || P.Cg % 2) return DCN_OK;
        const int mtiles = (P.M + TN - 1) / TN;
        // Which layers the 16-bit kernels take: those for which backward_weight16_kernel reads no more of the corners than the float32
        // kernels do on widened tensors, five to four.  It has two row tiles per workgroup at most (four would take 128 accumulator
        // registers beside its two channel tiles: one wavefront per SIMD), so more than 64 output channels sample everything once
        // per 64 of them, and channel segments that fill their 64-channel tiles badly waste the lanes' loads; it issues half as many per
        // channel (128 -> 128 channels in deformable groups of 32, 3-D: 2.5 ms against 1.2 + 0.15 for widening; 256 -> 256 in one
        // group, 2-D: 0.20 against 0.31).  backward_weight_split_kernel samples once for 128 output channels, but rounds the samples to the
        // storage format, which the widened operator does not: the line stands.
        c.MT = mtiles >= 2 ? 2 : 1;
        P.mchunks = (mtiles + c.MT - 1) / c.MT;
        P.nctiles = 0;
        int nct32 = 0;
        for (int gg = 0; gg < P.G; ++gg) {
            const int cg0 = gg * P.Cg, cg1 = cg0 + P.Cg;
            for (int dg = cg0 / P.cpg; dg <= (cg1 - 1) / P.cpg; ++dg) {
                const int cb = cg0 > dg * P.cpg ? cg0 : dg * P.cpg, ce = cg1 < (dg + 1) * P.cpg ? cg1 : (dg + 1) * P.cpg;
                P.nctiles += (ce - cb + CT - 1) / CT;
                nct32 += (ce - cb + TN - 1) / TN;
            }
        }
        {
            const long long loads16 = (long long)P.mchunks * P.nctiles, loads32 = (long long)((mtiles + 3) / 4) * nct32;
            if (4 * loads16 > 5 * loads32) return DCN_OK;
        }
        // position splits: about 2560 workgroups, as in the float kernel's plan
        const long long slabs = (long long)P.N * ((P.outV + TN - 1) / TN), other = (long long)P.kV * P.nctiles * P.mchunks;
        long long split = (2560 + other - 1) / other;
        const long long max_split = (slabs + WAVES - 1) / WAVES;
        if (split > max_split) split = max_split;
        if (split > 256) split = 256;
        if (split < 1) split = 1;
        P.nsplit = (int)split;
        if ((long long)P.nsplit * other > 0x7fffffffLL) return DCN_OK;
    }
    const size_t ibytes = align256((size_t)P.N * P.C_in * P.inV * sizeof(S));
    size_t obytes = align256((size_t)P.N * P.C_out * P.outV * sizeof(S));
    c.igroups = 0;
    c.gout = gout;
    if constexpr (sizeof(S) <= 4) {
        const size_t rbytes = align256(row_operand_bytes<S>(P.N, P.C_out, P.outV));
        const size_t used = ibytes + rbytes + (bias ? (size_t)P.N * last_strips(P.outV) * P.C_out * sizeof(T) : 0) + 256;
        const SplitPlan sp = split_plan<ND, S>(P, off != nullptr, ws && ws_bytes > used ? ws_bytes - used : 0);
        if (sp.nsplit) {
            obytes = rbytes;
            c.MT = sp.MT; c.LW = sp.LW; c.igroups = sp.igroups; P.mchunks = sp.mchunks; P.nsplit = sp.nsplit;
        }
    }
    const size_t pbytes = align256((size_t)P.nsplit * P.kV * P.C_out * P.Cg * sizeof(T));
    c.nsums = (int)(P.N * last_strips(P.outV));
    if (!ws || ws_bytes < ibytes + obytes + pbytes + (bias ? (size_t)c.nsums * P.C_out * sizeof(T) : 0)) return refuse(DCN_E_WORKSPACE, "workspace too small");
    if (declined) *declined = false;
    char* p = static_cast<char*>(ws);
    c.in_cl = reinterpret_cast<S*>(p);
    c.gout_cl = reinterpret_cast<S*>(p + ibytes);
    c.partial = reinterpret_cast<T*>(p + ibytes + obytes);
    c.sums = bias ? reinterpret_cast<T*>(p + ibytes + obytes + pbytes) : nullptr;
    prep.channels_last(in, c.in_cl, P.C_in, P.inV, P.N, nullptr);
    if (c.igroups) prep.rows(gout, c.gout_cl, P.C_out, P.outV, P.N, c.sums);
    else prep.channels_last(gout, c.gout_cl, P.C_out, P.outV, P.N, c.sums);
    return DCN_OK;
}

template <int ND, typename S>
int launch_bwd_weight_split(const WeightCall<float, S>& c, const S* off, hipStream_t s) {
    const Params& P = c.P;
    const dim3 grid((unsigned)((long long)c.igroups * P.mchunks * P.G * P.nsplit));
    if (trace_plans())
        fprintf(stderr, "dcn backward_weight, %s: %d row tiles, %d lanes to a tap, %d bytes of a corner to a lane, %d splits, grid %u\n",
                sizeof(S) == 4 ? "float32" : std::is_same<S, Bf16>::value ? "bfloat16" : "binary16", c.MT, c.LW, split_quad<ND, S>(P, c.MT, c.LW) ? 16 : 4, P.nsplit, grid.x);
    hipLaunchKernelGGL((split_kernel<ND, S>(P, c.MT, c.LW, !off)), grid, dim3(WG), 0, s, P, (const S*)c.in_cl, off, c.gout, reinterpret_cast<const typename Parts<S>::Vec*>(c.gout_cl), c.partial, (unsigned)c.igroups);
    return check_launch("backward_weight_split_kernel");
}

template <typename T, int ND, typename S>
int backward_weight_run(const WeightCall<T, S>& c, const S* off, T* gw, T* gb, bool accumulate, hipStream_t s) {
    const Params& P = c.P;
    if (c.igroups) {
        if constexpr (sizeof(T) == 4)
            if (int rc = launch_bwd_weight_split<ND, S>(c, off, s)) return rc;
    } else if constexpr (std::is_same<S, T>::value) {
        int rc;
        switch (c.MT) {
            case 1: rc = launch_bwd_weight<T, ND, 1>(c, off, s); break;
            case 2: rc = launch_bwd_weight<T, ND, 2>(c, off, s); break;
            default: rc = launch_bwd_weight<T, ND, 4>(c, off, s); break;
        }
        if (rc) return rc;
    } else {
        const int TN = Mma<float>::TN;
        const size_t lds = (size_t)WAVES * TN * (TN + 1) * sizeof(float);
        const dim3 grid((unsigned)P.nsplit * P.kV * P.nctiles * P.mchunks);
        if (c.MT == 2) hipLaunchKernelGGL((backward_weight16_kernel<ND, 2, S>), grid, dim3(WG), lds, s, P, (const S*)c.in_cl, off, (const S*)c.gout_cl, c.partial);
        else hipLaunchKernelGGL((backward_weight16_kernel<ND, 1, S>), grid, dim3(WG), lds, s, P, (const S*)c.in_cl, off, (const S*)c.gout_cl, c.partial);
        if (int rc = check_launch("backward_weight16_kernel")) return rc;
    }
    const size_t rows_x_cg = (size_t)P.C_out * P.Cg, total = rows_x_cg * P.kV;
    const unsigned rb = (unsigned)((total + 63) / 64 > 8192 ? 8192 : (total + 63) / 64), bb = gb ? ((unsigned)P.C_out + 3) / 4 : 0u;
    hipLaunchKernelGGL(reduce_weight_partials_kernel<T>, dim3(rb + bb), dim3(256), 0, s, (const T*)c.partial, gw, P.nsplit, P.kV, rows_x_cg, accumulate ? 1 : 0,
                       rb, (const T*)c.sums, gb, P.C_out, c.nsums);
    return check_launch("reduce_weight_partials_kernel");
}

#define INSTANTIATE(T, ND, S)                                                                                                                            \
    template int backward_weight_plan<T, ND, S>(const Params&, const S*, const S*, const S*, void*, size_t, bool, WeightCall<T, S>&, Prep&, bool*);           \
    template int backward_weight_run<T, ND, S>(const WeightCall<T, S>&, const S*, T*, T*, bool, hipStream_t);
INSTANTIATE(float, 2, float) INSTANTIATE(float, 3, float) INSTANTIATE(double, 2, double) INSTANTIATE(double, 3, double)
INSTANTIATE(float, 2, Bf16) INSTANTIATE(float, 3, Bf16) INSTANTIATE(float, 2, Fp16) INSTANTIATE(float, 3, Fp16)

}  // namespace dcn
