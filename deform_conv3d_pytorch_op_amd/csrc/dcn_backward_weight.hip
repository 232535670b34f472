// Backward pass to the weight: plans and launches.
#include "dcn_host.h"

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
int launch_bwd_weight(const Params& P, const T* in_cl, const T* off, const T* gout_cl, T* partial, hipStream_t s) {
    const int TN = Mma<T>::TN;
    const size_t lds = (size_t)WAVES * TN * (TN + 1) * sizeof(T);
    auto kern = backward_weight_kernel<T, ND, MT>;
    if (lds > 48 * 1024)
        if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds)) return rc;
    const dim3 grid((unsigned)P.nsplit * P.kV * P.nctiles * P.mchunks);
    hipLaunchKernelGGL(kern, grid, dim3(WG), lds, s, P, in_cl, off, gout_cl, partial);
    return check_launch("backward_weight_kernel");
}

template <typename T> size_t bww_workspace(const Params& P, int nsplit) {
    return align256((size_t)P.N * P.C_in * P.inV * sizeof(T)) + align256((size_t)P.N * P.C_out * P.outV * sizeof(T)) +
           align256((size_t)nsplit * P.kV * P.C_out * P.Cg * sizeof(T));
}

// Workspace of backward_weight: [ input channels-last | grad_output channels-last | partial tiles per split ]
template <typename T, int ND>
int backward_weight(const Geometry& g, const T* in, const T* off, const T* gout, T* gw, void* ws, size_t ws_bytes,
                    hipStream_t s) {
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !off || !gout || !gw) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    if (int rc = device_info(nullptr)) return rc;
    if ((long long)P.outV * P.C_out > (1ll << 31)) return fail(DCN_E_ARGUMENT, "one output sample exceeds 2^31 elements");
    // (the layout change of both operands is one launch with 2 * N slices along z)
    if (2 * (long long)P.N > 65535) return fail(DCN_E_ARGUMENT, "backward_weight: batch exceeds 32767");
    // the kernel addresses both operands by 32-bit byte offsets from the sample's base
    if ((unsigned long long)P.inV * P.C_in * sizeof(T) >= (1ull << 32) || (unsigned long long)P.outV * P.C_out * sizeof(T) >= (1ull << 32))
        return fail(DCN_E_ARGUMENT, "one sample of the input or of grad_output reaches 4 GiB");
    int MT;
    bww_plan<T>(P, MT, P.mchunks, P.nctiles, P.nsplit);
    const long long resident = MT == 1 ? bww_resident<T, ND, 1>() : MT == 2 ? bww_resident<T, ND, 2>() : bww_resident<T, ND, 4>();
    bww_plan<T>(P, MT, P.mchunks, P.nctiles, P.nsplit, resident);
    if ((long long)P.nsplit * P.kV * P.nctiles * P.mchunks > 0x7fffffffLL) return fail(DCN_E_ARGUMENT, "too many workgroups for one launch");
    const size_t ibytes = align256((size_t)P.N * P.C_in * P.inV * sizeof(T));
    const size_t obytes = align256((size_t)P.N * P.C_out * P.outV * sizeof(T));
    if (!ws || ws_bytes < bww_workspace<T>(P, P.nsplit)) return fail(DCN_E_WORKSPACE, "workspace too small");
    T* in_cl = static_cast<T*>(ws);
    T* gout_cl = reinterpret_cast<T*>(static_cast<char*>(ws) + ibytes);
    T* partial = reinterpret_cast<T*>(static_cast<char*>(ws) + ibytes + obytes);
    const dim3 tblock(32, 8);
    {
        const unsigned vmax = P.inV > P.outV ? P.inV : P.outV;
        const int cmax = P.C_in > P.C_out ? P.C_in : P.C_out;
        hipLaunchKernelGGL(to_channels_last_pair_kernel<T>, dim3((vmax + 31) / 32, (unsigned)(cmax + 31) / 32, 2u * (unsigned)P.N), tblock, 0, s,
                           in, in_cl, P.C_in, P.inV, gout, gout_cl, P.C_out, P.outV, P.N);
        if (int rc = check_launch("to_channels_last_pair_kernel")) return rc;
    }
    int rc;
    switch (MT) {
        case 1: rc = launch_bwd_weight<T, ND, 1>(P, in_cl, off, gout_cl, partial, s); break;
        case 2: rc = launch_bwd_weight<T, ND, 2>(P, in_cl, off, gout_cl, partial, s); break;
        default: rc = launch_bwd_weight<T, ND, 4>(P, in_cl, off, gout_cl, partial, s); break;
    }
    if (rc) return rc;
    const size_t rows_x_cg = (size_t)P.C_out * P.Cg, total = rows_x_cg * P.kV;
    const unsigned rb = (unsigned)((total + 63) / 64 > 8192 ? 8192 : (total + 63) / 64);
    hipLaunchKernelGGL(reduce_weight_partials_kernel<T>, dim3(rb), dim3(256), 0, s, partial, gw, P.nsplit, P.kV, rows_x_cg);
    return check_launch("reduce_weight_partials_kernel");
}

// backward_weight on the 16-bit tensors themselves (backward_weight16_kernel): channels-last copies of
// the input and of grad_output in their storage format, the offsets as they are, float partial tiles.
// Declines (nothing launched) where the kernel's 4-byte loads of channel pairs would not be aligned
// (an odd number of input channels, or segments -- intersections of convolution groups and deformable
// groups -- that start at odd channels) or the workspace is too small for it.
template <typename S, int ND>
int backward_weight_native16(const Params& Pin, const S* in, const S* off, const S* gout, float* fgw, void* ws, size_t ws_bytes,
                             hipStream_t s, bool* declined) {
    Params P = Pin;
    const int TN = Mma<float>::TN, CT = 2 * TN;
    *declined = true;
    if (P.C_in % 2 || P.cpg % 2 || P.Cg % 2) return DCN_OK;
    if ((unsigned long long)P.inV * P.C_in * sizeof(S) >= (1ull << 32) || (unsigned long long)P.outV * P.C_out >= (1ull << 32)) return DCN_OK;
    if (2 * (long long)P.N > 65535) return DCN_OK;
    const int mtiles = (P.M + TN - 1) / TN;
    // Two row tiles per workgroup at most (four would take 128 accumulator registers beside the two
    // channel tiles: one wavefront per SIMD), so more than 64 output channels sample everything once
    // per 64 of them, and channel segments that fill their 64-channel tiles badly waste the lanes'
    // loads.  Both kernels are bounded by their corner loads: this one issues half as many per
    // channel as the float32 kernel (four row tiles, 32-channel tiles), times the re-sampling and the
    // unused part of the tiles.  Where that comes to more than the float32 kernel's, that kernel on
    // widened tensors is the faster one (128 -> 128 channels in deformable groups of 32, 3-D: 2.5 ms
    // here against 1.2 + 0.15 for widening; 256 -> 256 in one group, 2-D: 0.20 here against 0.31).
    const int MT = mtiles >= 2 ? 2 : 1;
    P.mchunks = (mtiles + MT - 1) / MT;
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
    const size_t ibytes = align256((size_t)P.N * P.C_in * P.inV * sizeof(S));
    const size_t obytes = align256((size_t)P.N * P.C_out * P.outV * sizeof(S));
    const size_t pbytes = align256((size_t)P.nsplit * P.kV * P.C_out * P.Cg * sizeof(float));
    if (!ws || ws_bytes < ibytes + obytes + pbytes) return DCN_OK;
    *declined = false;
    S* in_cl = static_cast<S*>(ws);
    S* gout_cl = reinterpret_cast<S*>(static_cast<char*>(ws) + ibytes);
    float* partial = reinterpret_cast<float*>(static_cast<char*>(ws) + ibytes + obytes);
    {
        const unsigned vmax = P.inV > P.outV ? P.inV : P.outV;
        const int cmax = P.C_in > P.C_out ? P.C_in : P.C_out;
        hipLaunchKernelGGL(to_channels_last_pair_kernel<S>, dim3((vmax + 31) / 32, (unsigned)(cmax + 31) / 32, 2u * (unsigned)P.N), dim3(32, 8), 0, s,
                           in, in_cl, P.C_in, P.inV, gout, gout_cl, P.C_out, P.outV, P.N);
        if (int rc = check_launch("to_channels_last_pair_kernel")) return rc;
    }
    const size_t lds = (size_t)WAVES * TN * (TN + 1) * sizeof(float);
    const dim3 grid((unsigned)(P.nsplit * other));
    if (MT == 2) hipLaunchKernelGGL((backward_weight16_kernel<ND, 2, S>), grid, dim3(WG), lds, s, P, (const S*)in_cl, off, (const S*)gout_cl, partial);
    else hipLaunchKernelGGL((backward_weight16_kernel<ND, 1, S>), grid, dim3(WG), lds, s, P, (const S*)in_cl, off, (const S*)gout_cl, partial);
    if (int rc = check_launch("backward_weight16_kernel")) return rc;
    const size_t rows_x_cg = (size_t)P.C_out * P.Cg, total = rows_x_cg * P.kV;
    const unsigned rb = (unsigned)((total + 63) / 64 > 8192 ? 8192 : (total + 63) / 64);
    hipLaunchKernelGGL(reduce_weight_partials_kernel<float>, dim3(rb), dim3(256), 0, s, (const float*)partial, fgw, P.nsplit, P.kV, rows_x_cg);
    return check_launch("reduce_weight_partials_kernel");
}

#define INSTANTIATE(T, ND) template int backward_weight<T, ND>(const Geometry&, const T*, const T*, const T*, T*, void*, size_t, hipStream_t);
INSTANTIATE(float, 2) INSTANTIATE(float, 3) INSTANTIATE(double, 2) INSTANTIATE(double, 3)
#define INSTANTIATE16(S, ND) template int backward_weight_native16<S, ND>(const Params&, const S*, const S*, const S*, float*, void*, size_t, hipStream_t, bool*);
INSTANTIATE16(Bf16, 2) INSTANTIATE16(Bf16, 3) INSTANTIATE16(Fp16, 2) INSTANTIATE16(Fp16, 3)

}  // namespace dcn
