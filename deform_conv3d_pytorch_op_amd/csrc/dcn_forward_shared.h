// Forward kernel of the float32 and 16-bit operators for more than 64 output channels per group: the
// sampled columns of a block of 128 positions are made once, in LDS, for all of the workgroup's output channels.
//
// Where every wavefront samples into its own operands (forward_split_kernel), 256 output channels mean
// sampling everything twice and reading 12 KB of weights per 24 matrix instructions and wavefront:
// the L1 and its latency set the pace (256 -> 256 channels, 3x3, 25 088 positions: 0.277 ms; 0.239 here, with the matrix
// units of an occupied CU busy 46 % of the cycles, its vector ALUs 23 %).  Here eight wavefronts share the columns.  A phase is 32 reduction slots -- one tap pair, two groups of eight channels: each
// wavefront samples 32 positions of one group and writes its operand parts to LDS, and multiplies the
// previous phase's columns by its own row tiles, whose weights (each used by two wavefronts only) come
// straight from the L2 into registers a phase ahead.  Columns are double buffered, one barrier per phase;
// half of the wavefronts sample before they multiply and half after, so that the matrix and the
// vector / LDS work of a SIMD's two wavefronts fall next to each other.
#pragma once
#include "dcn_forward_split.h"

namespace dcn {

constexpr int SHARED_COLS = 4;             // column tiles (of 32 positions) of a workgroup
constexpr int SHARED_WAVES = 8;
template <typename S> __host__ __device__ inline constexpr size_t shared_column_bytes() {      // both buffers
    return (size_t)2 * 2 * SHARED_COLS * Parts<S>::NP * 1024 < 2 * SHARED_COLS * 64 * FG * 4 ? (size_t)2 * SHARED_COLS * 64 * FG * 4
                                                                                             : (size_t)2 * 2 * SHARED_COLS * Parts<S>::NP * 1024;
}

// RT row tiles (4 or 8) of a unit; grid and splits as forward_split_kernel; dynamic LDS = columns, then
// cchunk * hstride * sizeof(S) bytes of halo with cchunk a multiple of eight.
template <int ND, int RT, typename S>
__global__ __launch_bounds__(SHARED_WAVES * 64, 2) void forward_shared_kernel(Params P, PlanSet alts, const unsigned* __restrict__ sel,
                                                           const S* __restrict__ in, const S* __restrict__ off,
                                                           const typename Parts<S>::Elem* __restrict__ Wq, const S* __restrict__ W,
                                                           const S* __restrict__ bias, S* __restrict__ out, float* __restrict__ part, Div csplit,
                                                           unsigned whole, TailSplit ts) {
    touch_arguments<sizeof(Params) + sizeof(PlanSet) + 96>();
    HaloPlan H;
    if (!chosen_halo(P, alts, sel, H)) return;          // another launch runs the chosen plan
    using PT = Parts<S>;
    using MM = Mma<float>;
    typedef typename PT::Vec Vec;
    typedef typename PT::Elem Elem;
    constexpr int TN = 32, NP = PT::NP, CT = SHARED_COLS, WGS = SHARED_WAVES * 64;
    constexpr int RW = RT / 4, CW = 2;                  // row and column tiles of a wavefront: four wavefronts along rows, two along columns
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int sNonFinite, sRedo;
    Vec* sB = reinterpret_cast<Vec*>(smem_raw);                                         // [buffer][group][column tile][part][lane]
    typedef typename HaloCell<S>::Vec Cell;
    Cell* sIn = reinterpret_cast<Cell*>(smem_raw + shared_column_bytes<S>());
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % TN, q = lane / TN;
    const int rw = wave & 3, cwv = wave >> 2;           // this wavefront's row tiles and column tiles of the product
    const int ct = wave & 3, half = wave >> 2;          // what it samples: column tile, group of the phase
    const ForwardUnit U = forward_unit(H.cchunk, csplit, whole, ts);
    const unsigned rest = U.wg / P.mchunks;
    const int g = rest % P.G, mchunk = U.wg - rest * P.mchunks;
    TileGeo<ND> tg;
    tile_decode<ND>(P, H, rest / P.G, tg);
    const int n = tg.n;
    int ib[ND];
    unsigned pos;
    bool valid;
    {
        int o[ND];
        valid = tile_position<ND>(P, tg, ct * TN + j, o, pos);
#pragma unroll
        for (int a = 0; a < ND; ++a) ib[a] = o[a] * P.stride[slot<ND>(a)] - P.pad[slot<ND>(a)];
    }
    typename MM::Acc acc[CW * RW];                      // [column tile][row tile]
    const int ntg = (P.kV + 1) / 2;
    const unsigned mtiles = P.Mp / TN;
    const unsigned per_slab = (unsigned)ntg * mtiles * NP * 64;        // operands (16 bytes) of a slab
    const unsigned row = (unsigned)H.hext[2], plane = ND == 3 ? (unsigned)(H.hext[1] * H.hext[2]) : 0u;
    const unsigned a_lane = (unsigned)lane * 16;
    const int cg0 = g * P.Cg, cg1 = cg0 + P.Cg;
    if (threadIdx.x == 0) sRedo = 0;                    // ordered before the checks by the barriers of the first chunk

    auto work = [&](auto exact_tag) {
        constexpr bool exact = decltype(exact_tag)::value;
#pragma unroll
        for (int i = 0; i < CW * RW; ++i) acc[i] = acc_zero<float>();
        int chunk_no = 0;
        const int dg_last = (cg1 - 1) / P.cpg;          // (in the loop's condition, with its loop unrolled, it sends the accumulators through scratch memory)
#pragma unroll 1
        for (int dg = cg0 / P.cpg; dg <= dg_last; ++dg) {
            const int cb = max(cg0, dg * P.cpg), ce = min(cg1, (dg + 1) * P.cpg);
            const S* off_dg = off + ((size_t)n * P.DG + dg) * P.kV * ND * P.outV;
            for (int cc0 = cb; cc0 < ce; cc0 += U.cch) {
                const int turn = chunk_no++;
                if (U.split && turn % U.cs != U.cz) continue;                  // another workgroup's chunk (uniform)
                const int nch = min(U.cch, ce - cc0);
                const int ngrp = (nch + FG - 1) / FG, npair = (ngrp + 1) / 2;
                const S* chan0 = in + ((size_t)n * P.C_in + cc0) * P.inV;      // workgroup-uniform
                const Elem* wchunk = Wq + ((size_t)chunk_slot<FG>(P.cpg, P.Cg, cc0) * per_slab + ((size_t)mchunk * RT + rw * RW) * NP * 64) * FG;
                float ofs[ND];
                load_pair_offsets<ND, S>(P, off_dg, 0, q, pos, ofs, off == nullptr);
                if (exact && threadIdx.x == 0) sNonFinite = 0;
                __syncthreads();                                               // readers of the previous chunk are done
                if (stage_halo<ND, WGS, exact, S>(P, H, tg, chan0, nch, sIn)) sNonFinite = 1;
                Vec a8[2][RW][NP];
                // weights of this wavefront's row tiles for tap pair tgi and the groups 2 * gp, 2 * gp + 1
                auto load_a = [&](int tgi, int gp) {
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks) {
                        const char* wp = reinterpret_cast<const char*>(wchunk + ((size_t)min(2 * gp + ks, ngrp - 1) * per_slab + (size_t)tgi * mtiles * NP * 64) * FG);
#pragma unroll
                        for (int r = 0; r < RW; ++r)
#pragma unroll
                            for (int k = 0; k < NP; ++k) a8[ks][r][k] = *reinterpret_cast<const Vec*>(wp + (r * NP + k) * 1024 + a_lane);
                    }
                };
                if constexpr (!(exact && sizeof(S) == 4)) load_a(0, 0);
                __syncthreads();
                const bool rim_far = exact && sNonFinite != 0;                 // uniform, see forward_split_kernel
                int k0[ND];                            // kernel coordinates of the next tap pair
#pragma unroll
                for (int a = 0; a < ND; ++a) k0[a] = 0;
                SplitTap<ND> t;
                bool any_far = false;
                // samples this wavefront's share of phase (tgi, gp) into buffer b
                auto produce = [&](int tgi, int gp, int b) {
                    if (gp == 0) {
                        int k1[ND];
#pragma unroll
                        for (int a = 0; a < ND; ++a) k1[a] = k0[a];
                        next_tap<ND>(P, k1);
                        split_geometry<ND>(P, H, tg, ib, q, k0, k1, ofs, valid && tgi * 2 + q < P.kV, rim_far, t);
                        any_far = __any(t.far);
                        next_tap<ND>(P, k1);
#pragma unroll
                        for (int a = 0; a < ND; ++a) k0[a] = k1[a];
                        load_pair_offsets<ND, S>(P, off_dg, min(tgi + 1, ntg - 1), q, pos, ofs, off == nullptr);
                    }
                    const int grp = 2 * gp + half;
                    if (grp >= ngrp) return;
                    float val[FG];
                    group_sum8<ND, S>(sIn, t.base, grp, nch, H.hstride, row, plane, t.cw, val);
                    if (__builtin_expect(any_far, 0)) far_values<ND, S>(P, t, chan0, grp * FG, nch, val);
                    if constexpr (exact) {
                        float* dst = reinterpret_cast<float*>(sB) + ((size_t)(half * CT + ct) * 64 + lane) * FG;
#pragma unroll
                        for (int e = 0; e < FG; ++e) dst[e] = (t.near || t.far) && grp * FG + e < nch ? val[e] : 0.f;
                    } else {
                        Vec b8[NP];
                        PT::split(val, b8);
                        Vec* dst = sB + ((size_t)((b * 2 + half) * CT + ct) * NP) * 64 + lane;
#pragma unroll
                        for (int k = 0; k < NP; ++k) dst[k * 64] = b8[k];
                    }
                };
                // this wavefront's row tiles times its column tiles of buffer b
                auto consume = [&](int tgi, int gp, int b) {
                    const bool two = 2 * gp + 1 < ngrp;                        // uniform
                    if constexpr (exact) {
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks)
                            if (ks == 0 || two)
#pragma unroll
                                for (int c = 0; c < CW; ++c) {
                                    const float* src = reinterpret_cast<const float*>(sB) + ((size_t)(ks * CT + cwv * CW + c) * 64 + lane) * FG;
                                    float val[FG];
#pragma unroll
                                    for (int e = 0; e < FG; ++e) val[e] = src[e];
                                    mma_exact<S, RW>(P, W, g, (mchunk * RT + rw * RW) * TN + j, tgi * 2 + q, (size_t)(cc0 - cg0 + (2 * gp + ks) * FG), a8[ks], val, true,
                                                     nch - (2 * gp + ks) * FG, acc + c * RW);
                                }
                    } else {
                        // all columns of the phase are requested before the first matrix instruction
                        // (left alone, the compiler reads each just before its use and waits four times)
                        Vec b8[2][CW][NP];
#pragma unroll
                        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                            for (int c = 0; c < CW; ++c)
#pragma unroll
                                for (int k = NP - 1; k >= 0; --k) b8[ks][c][k] = sB[((size_t)((b * 2 + ks) * CT + cwv * CW + c) * NP + k) * 64 + lane];
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int c = 0; c < CW; ++c) mma_parts<S, RW>(a8[0], b8[0][c], acc + c * RW);
                        if (two) {
#pragma unroll
                            for (int c = 0; c < CW; ++c) mma_parts<S, RW>(a8[1], b8[1][c], acc + c * RW);
                        }
                    }
                };
                int tgi = 0, gp = 0, b = 0;
                produce(0, 0, 0);
                __syncthreads();
                while (true) {
                    const int gn = gp + 1 < npair ? gp + 1 : 0, tn = gn ? tgi : tgi + 1;
                    const bool more = tn < ntg;                                // uniform
                    if constexpr (exact) {
                        consume(tgi, gp, 0);
                        if (!more) break;
                        if constexpr (sizeof(S) == 2) load_a(tn, gn);
                        __syncthreads();
                        produce(tn, gn, 0);
                    } else {
                        if (more && half == 0) produce(tn, gn, b ^ 1);
                        consume(tgi, gp, b);
                        if (!more) break;
                        load_a(tn, gn);
                        if (half != 0) produce(tn, gn, b ^ 1);
                    }
                    tgi = tn;
                    gp = gn;
                    b ^= 1;
                    __syncthreads();
                }
            }
        }
    };
    work(std::false_type{});

    bool ok[CW];
    unsigned opos[CW];
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        int o[ND];
        ok[c] = tile_position<ND>(P, tg, (cwv * CW + c) * TN + j, o, opos[c]);
        if (ok[c] && !results_stand<RW, S>(acc + c * RW)) sRedo = 1;
    }
    __syncthreads();
    if (__builtin_expect(sRedo, 0)) work(std::true_type{});

    const size_t sample = (size_t)n * P.C_out * P.outV;
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            const int rt = rw * RW + r, m0 = (mchunk * RT + rt) * TN;
            if (U.split && whole > 0) {                // [split workgroup][RT * TN rows][CT * TN positions]
                float* dst = part + ((size_t)U.pslot * (RT * TN) + rt * TN + q * 4) * (CT * TN) + (cwv * CW + c) * TN + j;
#pragma unroll
                for (int e = 0; e < MM::NACC; ++e) dst[MM::row(e, 0) * (CT * TN)] = acc[c * RW + r][e];
            } else if (ok[c]) {
                if (U.split) store_tile<float, S>(P, part + (size_t)U.cz * P.N * P.C_out * P.outV + sample, nullptr, g, m0, q, opos[c], acc[c * RW + r]);
                else store_tile<S, S>(P, out + sample, bias, g, m0, q, opos[c], acc[c * RW + r]);
            }
        }
}

}  // namespace dcn
