// Plain convolution of float32 in 2-D (offsets that are all zero): forward pass, and backward pass to the input at stride 1.
//
//   out[n][g*M + m][pos] = sum_{cl,tap} W[g*M+m][cl][tap] * in[n][g*Cg+cl][pos * stride - pad + tap * dil]  (+ bias)
//
// replaces im2col + the per-group Sgemm of the reference (conv2d/lib/conv2d_cuda.cpp:77-290, conv2d/lib/conv2d_cuda_kernel.cu:25-169).
//
// forward_split_kernel with a null offset works out the geometry of every (tap, position), weighs four corners of which three have weight
// zero, and splits every sample into its bfloat16 parts once per tap.  Here a value is split once, on its way into LDS, where a voxel's
// parts lie as the operands want them -- [part][voxel][channel] -- so that a step of the contraction is three 16-byte LDS reads at a tap's
// fixed distance, the weights from L2 (a few steps ahead, in the order of pack_split_weight_kernel) and six matrix instructions a row tile.
// A workgroup has two position tiles (a block of 64 positions) and MW wavefronts along the rows, RW row tiles each.
// Small layers: the matrix instructions of 64 -> 64 channels, 3x3, 8 x 56 x 56 take 5 us of the device, a workgroup's first instructions and
// loads as long again.  us of a forward call with the packing of its weights, on the former kernels -> here: that layer 36 -> 26 (a training step 102 -> 90),
// 100 -> 100, 5x5, 4 x 60 x 60: 131 -> 69; 512 -> 512, 8 x 28 x 28: 272 -> 237.
// Sums: every matrix instruction rounds what it adds to, and cuts products off towards minus infinity below its last places; a result that went through six of them in
// each of some hundred steps was up to twice as far from float64 as that of the kernels before, whose chains are shorter where they share a position.  Here the products of
// a step start from zero, and their sum is added to the result while the next one's are formed; every second slab of channels lies in LDS with its sign turned round, and so
// do the sums that come of it.  Error against float64, 2-norm, of 260 layers over the kernels before: 0.41 on average, at worst 0.81, where the sum through all steps had
// 0.99 and 1.98.  The additions are placed between the matrix instructions (the scheduler's own order, all of them after the first, cost layers of two row tiles to a
// wavefront 5 %): 150 layers 0.986 of the time of the sum through all steps, at worst 1.066.
#pragma once
#include "dcn_forward_split.h"

namespace dcn {

constexpr int PLAIN_COLS = 2;                           // position tiles of a workgroup
constexpr size_t MAX_PLAIN_LDS = 160 * 1024 - 256;      // dynamic LDS of a workgroup
// operands of a voxel in a part's plane: an odd number, so that eight voxels in a row lie in different LDS banks
__host__ __device__ inline constexpr int plain_row(int channels) { return (channels / FG) | 1; }
__host__ inline size_t plain_lds(int hvol, int channels) { return (size_t)Parts<float>::NP * hvol * plain_row(channels) * 16; }

// Wavefronts along the rows, row tiles of each, chunks of rows.  Two row tiles to a wavefront, for half the staging and half the reads of values, where that makes no more
// rows than one does, and of a single tap, which is all staging, up to a quarter more.  293 layers of nine to twelve and of seventeen to twenty row tiles, us of the forward call
// with two : one -- 92 -> 339, 3x3, 82 x 112, 88 : 53; 225 -> 379, 3x3, two samples of 18 x 210, 195 : 113; 20 -> 591, 3x3, 16 x 17 x 16, 31 : 21; on average 1.22 : 1 and, from
// seventeen on, 1.07 : 1, at worst 0.90 : 1; single taps 1.09 : 1 up to twelve, from seventeen on 0.95 : 1 (13 -> 592, four of 106 x 219, 76 : 88).
struct PlainRows { int mw, rw, mchunks; };
inline PlainRows plain_rows(int M, int taps) {
    const int tiles = (M + 31) / 32, four = (tiles + 3) / 4 * 4, eight = (tiles + 7) / 8 * 8;
    PlainRows r;
    r.mw = tiles > 2 ? 4 : tiles;
    r.rw = tiles > 4 && (eight == four || (taps == 1 && eight * 4 <= four * 5)) ? 2 : 1;
    r.mchunks = (tiles + r.mw * r.rw - 1) / (r.mw * r.rw);
    return r;
}

// Channels at a time, `most` of them at most: two workgroups to a CU.  Those of one row tile are two wavefronts each: four, if there are so many, unless it leaves less than 24 channels.
// 81 such layers, us of the forward call with two : with four, 1.22 : 1 on average: 276 -> 15, 3x3, dilation 2, eight samples of 81 x 62, 140 : 86; 157 -> 8, 5x5, sixteen of 89 x 29,
// 153 : 95; 62 -> 25, 5x5, dilation 2, sixteen of 181 x 9, 76 : 47.
inline int plain_channels(const PlainRows& r, long long workgroups, int most, int hvol, int cus) {
    int c = most;
    while (c > FG && plain_lds(hvol, c) > MAX_PLAIN_LDS / 2) c -= FG;
    if (r.mw == 1 && workgroups > 2 * (long long)cus)
        while (c > 3 * FG && plain_lds(hvol, c) > MAX_PLAIN_LDS / 4) c -= FG;
    return c;
}

// Which layers take it.  A wavefront goes through the steps of sixteen reduction slots one after the other, 0.23 us to each (0.33 beside three others along the rows, 0.66 with
// two row tiles) whatever the device does, and 0.5 to 0.8 us to each of its thread's cells of the halo, of eight channels; the kernels of the deformable layer share a
// position or its channels among up to sixteen wavefronts.  So enough workgroups take it always and fewer only short chains: `steps` and 2.5 for every cell, up to a line that
// rises with the workgroups.  2400 layers, us of the forward call on those kernels : here, always here 1.26 times as fast on average, by these lines and by the faster of the two
// 1.28.  Refused: one row tile -- 256 -> 16, 1x1, two samples of 60 x 60, 14.1 : 22.1; 64 -> 32, 3x3, two of 60 x 60, 13.7 : 19.3 --, two -- 64 -> 64, 3x3, two
// of 60 x 60, 16.5 : 19.1; 129 -> 56, 1x1, stride 2, sixteen of 29 x 18, 15.1 : 21.0 --, eight -- 24 -> 256, 5x5, 56 x 56, 30.7 : 34.9; 64 -> 273, 3x3, 28.8 : 44.4 --, long chains of few
// wavefronts -- 512 -> 32, 3x3, 25 x 24 x 24, 68 : 118.  Taken: 64 -> 64, 3x3, 56 x 56, 21.9 : 20.4; 16 -> 128, 3x3, two of 40 x 40, 20.3 : 13.8; 256 -> 128, sixteen of 28 x 28, 108 : 79;
// 59 -> 131, 3x3, eight of 24 x 23, 63 : 35; at worst 38 : 42 (251 -> 196, 1x1, stride 2, eight of 44 x 51).
inline bool plain_pays(const PlainRows& r, long long workgroups, int channels, int taps, int hvol, int cus) {
    const int slabs = (channels + FG - 1) / FG, steps = slabs * ((taps + 1) / 2);
    const long long waves = workgroups * PLAIN_COLS * r.mw;
    if (waves * 2 >= 11 * (long long)cus) return true;
    if (steps > 40 || waves * 4 < 3 * (long long)cus) return false;
    const double load = steps + 2.5 * slabs * hvol / (64.0 * PLAIN_COLS * r.mw), per_cu = (double)workgroups / cus;
    if (r.mw == 1) return load <= 10 + 20 * per_cu;
    // (from 64 channels on the other kernels split those of so few blocks into eight parts, which a further launch joins)
    if (r.mw == 2) return load <= 26 || load <= 10 + 50 * per_cu || (channels >= 64 && taps > 1 && per_cu <= 0.25);
    if (r.rw == 1) return load <= 60;
    return steps <= 20 || (per_cu >= 0.25 && slabs > 3);
}

// Grid: N * tiles * G * mchunks workgroups of PLAIN_COLS * MW wavefronts; P.cchunk a multiple of eight.  AHEAD: steps that weights are read ahead by, as many as leave
// two workgroups to a CU (eight wavefronts each, of 128 registers, where four are along the rows): see plain_kernel.
template <int RW, int AHEAD>
__global__ __launch_bounds__(AHEAD == 4 ? 256 : 512, AHEAD == 4 ? 2 : 4) void plain_conv_kernel(Params P, const float* __restrict__ in, const Parts<float>::Vec* __restrict__ Wq,
                                                         const float* __restrict__ W, const float* __restrict__ bias, float* __restrict__ out) {
    touch_arguments<sizeof(Params) + 32>();
    using PT = Parts<float>;
    using MM = Mma<float>;
    typedef PT::Vec Vec;
    constexpr int TN = 32, NP = PT::NP, UN = AHEAD > 2 ? AHEAD : 2;
    constexpr int NA = AHEAD == 4 ? 2 : RW;             // results being summed up: of one row tile, two where there are registers for them
    extern __shared__ __align__(16) unsigned char smem_raw[];
    Vec* sX = reinterpret_cast<Vec*>(smem_raw);         // [part][voxel][slab of eight channels]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), WGS = (int)blockDim.x;
    const int j = lane % TN, q = lane / TN;
    const int pt = wave % PLAIN_COLS, mw = wave / PLAIN_COLS, MW = WGS / (64 * PLAIN_COLS);
    const unsigned unit = xcd_contiguous(blockIdx.x, gridDim.x), rest = unit / P.mchunks;
    const int g = rest % P.G, mchunk = (int)(unit - rest * (unsigned)P.mchunks.d);
    HaloPlan H;
    H.mlo[1] = H.mlo[2] = 0;
    TileGeo<2> tg;
    tile_decode<2>(P, H, rest / P.G, tg);
    int o[2];
    unsigned pos;
    bool valid = tile_position<2>(P, tg, pt * TN + j, o, pos);
    const int row = P.hext[2], hvol = P.hvol;
    const int at = (o[0] * P.stride[1] - P.pad[1] - tg.hb[0]) * row + o[1] * P.stride[2] - P.pad[2] - tg.hb[1];      // the position's voxel at tap 0
    const int cg0 = g * P.Cg, cg1 = cg0 + P.Cg, ntg = (P.kV + 1) / 2;
    const unsigned mtiles = P.Mp / TN, tile0 = (unsigned)(mchunk * MW + mw) * RW;
    const unsigned a_tg = mtiles * NP * 64, per_slab = (unsigned)ntg * a_tg;      // operands
    const float inv = __builtin_amdgcn_rcpf((float)hvol), inv_row = __builtin_amdgcn_rcpf((float)row);
    const int rs = plain_row(P.cchunk);

    MM::Acc acc[NA], part[2] = {acc_zero<float>(), acc_zero<float>()};      // results; sums of a step, one being formed and one to be added
#pragma unroll
    for (int r = 0; r < NA; ++r) acc[r] = acc_zero<float>();
    auto add = [&](int r, const MM::Acc& sum, float sign) {
#pragma unroll
        for (int i = 0; i < MM::NACC; ++i) acc[r][i] = fmaf(sum[i], sign, acc[r][i]);
    };
#pragma unroll 1
    for (int cc0 = cg0; cc0 < cg1; cc0 += P.cchunk) {
        const int nch = min(P.cchunk, cg1 - cc0), nsl = (nch + FG - 1) / FG;
        const float* chan0 = in + ((size_t)P.C_in * tg.n + cc0) * P.inV;
        // Steps: tap pairs, and the slabs of each.  Weights of this wavefront's row tiles, AHEAD steps ahead.
        const Vec* wp = Wq + (size_t)chunk_slot<FG>(P.cpg, P.Cg, cc0) * per_slab + tile0 * (NP * 64) + lane;
        const int steps = nsl * ntg;
        Vec a8[AHEAD][RW][NP];
        int asl = 0, atg = 0;
        unsigned lat = 0;
        auto load_a = [&](int u) {
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int k = 0; k < NP; ++k) a8[u][r][k] = wp[lat + (r * NP + k) * 64];
            lat += per_slab;
            if (++asl == nsl) {
                asl = 0;
                atg = min(atg + 1, ntg - 1);            // (past the last step the last pair again, for nothing)
                lat = (unsigned)atg * a_tg;
            }
        };
        if (cc0 > cg0) __syncthreads();                 // readers of the last channels are done
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) load_a(u);
        const int items = nsl * hvol;
#pragma unroll 2
        for (int it = (int)threadIdx.x; it < items; it += WGS) {
            const int sl = (int)(((float)it + 0.5f) * inv), v = it - __mul24(sl, hvol);
            const int vh = (int)(((float)v + 0.5f) * inv_row), ch = vh + tg.hb[0], cw = v - __mul24(vh, row) + tg.hb[1];
            const bool there = (unsigned)ch < (unsigned)P.in[1] && (unsigned)cw < (unsigned)P.in[2];
            const unsigned to = there ? (unsigned)ch * (unsigned)P.in[2] + (unsigned)cw : 0u;
            float x[FG];
#pragma unroll
            for (int e = 0; e < FG; ++e) x[e] = chan0[(size_t)min(sl * FG + e, nch - 1) * P.inV + to];
#pragma unroll
            for (int e = 0; e < FG; ++e) x[e] = __uint_as_float(__float_as_uint(there && sl * FG + e < nch ? x[e] : 0.f) ^ (unsigned)sl << 31);
            Vec p[NP];
            PT::split(x, p);
#pragma unroll
            for (int k = 0; k < NP; ++k) sX[((size_t)k * hvol + v) * rs + sl] = p[k];
        }
        __syncthreads();
        Vec b8[2][NP];
        float sign[2], last = 1.f;                      // of the sums of a step
        int k0[2] = {0, 0}, bsl = 0, btg = 0;
        const Vec* bp = nullptr;
        auto pair = [&]() {                             // this lane's voxel at tap pair btg
            int k1[2] = {k0[0], k0[1]};
            next_tap<2>(P, k1);
            int t0 = k0[0] * P.dil[1] * row + k0[1] * P.dil[2], t1 = k1[0] * P.dil[1] * row + k1[1] * P.dil[2];
            t1 = 2 * btg + 1 < P.kV ? t1 : t0;          // (its weights are zero)
            bp = sX + (size_t)(at + (q ? t1 : t0)) * rs;
            next_tap<2>(P, k1);
            k0[0] = k1[0]; k0[1] = k1[1];
        };
        const size_t plane = (size_t)hvol * rs;
        auto load_b = [&](int u) {
#pragma unroll
            for (int k = 0; k < NP; ++k) b8[u][k] = bp[k * plane];
            ++bp;
            sign[u] = bsl & 1 ? -1.f : 1.f;
            if (++bsl == nsl) {
                bsl = 0;
                if (++btg < ntg) pair();
                else bp -= nsl;
            }
        };
        pair();
        load_b(0);
        for (int s = 0; s < steps; s += UN) {
#pragma unroll
            for (int u = 0; u < UN; ++u)
                if (s + u < steps) {                    // (uniform)
                    load_b((u + 1) & 1);
#pragma unroll
                    for (int r = 0; r < RW; ++r) {
                        const int i = u * RW + r;
                        part[i & 1] = acc_zero<float>();
                        mma_parts<float, 1>(a8[u % AHEAD] + r, b8[u & 1], part + (i & 1));
                        add(RW == 1 ? u / 2 % NA : 1 - r, part[(i + 1) & 1], r ? sign[u & 1] : last);
                    }
                    last = sign[u & 1];
                    load_a(u % AHEAD);
#pragma unroll
                    for (int i = 0; i < 6 * RW; ++i) {  // a matrix instruction, three others, ...
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        add(RW - 1, RW == 1 && (steps & 1) ? part[0] : part[1], last);
        part[1] = acc_zero<float>();
    }
#pragma unroll
    for (int r = RW; r < NA; ++r) acc[0] += acc[r];
    // (lane and position once more: kept through the steps they are spilled)
    int me = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(me));
    const int mj = me % TN, mq = me / TN;
    valid = tile_position<2>(P, tg, pt * TN + mj, o, pos);
    // Results that the parts may have cost bits (see dcn_forward_split.h): once more on the float32 instructions, from the values themselves.
    if (__builtin_expect(__any(valid && !results_stand<RW, float>(acc)), 0)) {
#pragma unroll
        for (int r = 0; r < RW; ++r) acc[r] = acc_zero<float>();
        int kk[2] = {0, 0};
#pragma unroll 1
        for (int tap = 0; tap < P.kV; ++tap) {
            const int ch = o[0] * P.stride[1] - P.pad[1] + kk[0] * P.dil[1], cw = o[1] * P.stride[2] - P.pad[2] + kk[1] * P.dil[2];
            const bool there = valid && (unsigned)ch < (unsigned)P.in[1] && (unsigned)cw < (unsigned)P.in[2];
            const float* x = in + (size_t)P.C_in * P.inV * tg.n + (there ? (unsigned)ch * (unsigned)P.in[2] + (unsigned)cw : 0u);
#pragma unroll 1
            for (int cl = 0; cl < P.Cg; cl += 2) {
                const int c = min(cl + mq, P.Cg - 1);
                const float xv = x[(size_t)(cg0 + c) * P.inV], b = there && cl + mq < P.Cg ? xv : 0.f;
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    const int m = (int)(tile0 + r) * TN + mj;
                    const float wv = weight_at<float>(P, W, g, min(m, P.M - 1), (size_t)c, tap);
                    acc[r] = MM::mma(m < P.M && cl + mq < P.Cg ? wv : 0.f, b, acc[r]);
                }
            }
            next_tap<2>(P, kk);
        }
    }
    if (!valid) return;
#pragma unroll
    for (int r = 0; r < RW; ++r)
        store_tile<float, float>(P, out + (size_t)P.C_out * P.outV * tg.n, bias, g, (int)(tile0 + r) * TN, mq, pos, acc[r]);
}

using PlainKern = void (*)(Params, const float*, const Parts<float>::Vec*, const float*, const float*, float*);
inline PlainKern plain_kernel(const PlainRows& r) { return r.rw == 2 ? plain_conv_kernel<2, 1> : r.mw == 4 ? plain_conv_kernel<1, 2> : plain_conv_kernel<1, 4>; }

}  // namespace dcn
