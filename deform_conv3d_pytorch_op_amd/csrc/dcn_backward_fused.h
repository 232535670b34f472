// Backward pass to input and offset of the float32 and 16-bit operators, one kernel: grad columns on the 16-bit
// matrix instructions, their scatter into LDS cells (grad_input) and the coordinate gradient (grad_offset).
//
//   gcol[c][tap][pos] = sum_m W[m][c][tap] * grad_output[m][pos]
//   grad_input[voxel] += corner weight * gcol,   grad_offset[tap][axis][pos] = sum_c gcol * d sample / d coordinate
//
// replaces the grad-column Sgemm, deformable_col2im_input and deformable_col2im_offset of the reference
// (deform3d/lib/deform_conv3d_cuda.cpp:213-220, deform3d kernel.cu:229-296 and :386-483 incl. the out-of-range branches
// :470-481; deform2d_double kernel.cu:201-238, :309-366).
//
// A workgroup owns a block of NPT * 32 output positions and works through CCH input channels at a time: their
// values over the block's halo and the cells that collect their gradient sit in LDS.  The rows of a 32 x 32 result tile
// are (tap, channel) pairs, 32 / CCH taps of the CCH channels, so that a lane receives all channels of a tap at
// its position: lane group q the taps q, q + 2, ... of the tile.  It then walks its registers, one tap slot at a time:
// geometry, eight (four) corner reads per four channels, the sums for grad_offset, the adds to the cells.
//
// Sixteen wavefronts: 16 / NPT of them share 32 positions and take every (16 / NPT)th tile of a chunk, PT tiles to a
// contraction.  What a chunk costs is LDS work (a tap slot of eight channels in 3-D: 32 64-bit adds of 7 ns and 16 16-byte reads
// of 5 ns, two thirds of it bank conflicts of random voxels), vector work of about the same length, and the phases between the
// barriers: flush, staging, first loads.  Wavefronts in flight are what overlaps them, so a lane has to do with 128 registers:
// nothing of an operand stays in them past its contraction, and grad_output comes from memory every time, in the operand order
// that the preparing launch has brought it to (split_grad_output).  Vector memory operations complete in order, so the next
// chunk's contraction and input loads go out before a chunk's flush, whose atomics they would otherwise wait for (64 -> 64
// channels, 3x3x3, 200 704 positions: 1.41 -> 1.31 ms).
// Against the eight wavefronts, grad_output in registers and float32 matrix instructions that float32 layers had before, ms per call of
// backward_input_offset with its preparation: that layer 1.34 -> 1.31, in bfloat16 1.29 -> 1.10; 128 -> 128 in deformable groups of 32,
// stride 1 2 2, 100 352 positions 2.93 -> 2.49, in bfloat16 2.26 -> 2.09; 2-D 256 -> 256, 25 088 positions 0.61 -> 0.42, in binary16
// 0.64 (on widened tensors) -> 0.23; 512 -> 512 in two groups, 3136 positions 0.193 -> 0.145.  It pays for it with traffic: grad_output in
// operand order, half as much again as the tensor, is written once and read past the L2 by every block, for each chunk and as far as the
// L2 lets go of it for each tile (2-D 256 -> 256 0.20 -> 0.84 GB a call, 64 -> 64 in 3-D 2.4 -> 4.6 GB).  Tried and slower or no
// faster: the weights of a step shared through the LDS (the wavefronts then multiply together and scatter together), operands of the contraction a
// step ahead in registers of their own (grad_output's in 3-D float32 0 to 0.3 %, with the weights' 3 % slower, in 2-D 4 to 6 %: they spill), two workgroups of
// eight wavefronts per CU (2-D: 1 to 5 % faster on large layers, 13 % slower on 3600 positions), two tiles to a contraction in 3-D.
#pragma once
#include "dcn_forward_split.h"

namespace dcn {

// Row i of a tile: accumulator register r of lane group qq (Mma<float>::row) holds tap 2 * (r / CCH) + qq, channel r % CCH.
template <int CCH> __host__ __device__ inline constexpr int fused_row_tap(int i) { return 2 * (((i >> 3) * 4 + (i & 3)) / CCH) + ((i >> 2) & 1); }
template <int CCH> __host__ __device__ inline constexpr int fused_row_channel(int i) { return ((i >> 3) * 4 + (i & 3)) % CCH; }
__host__ __device__ inline int fused_steps(int M) { return (M + 15) / 16; }                   // of 16 output channels
__host__ __device__ inline int fused_tiles(int kV, int cch) { return (kV + 32 / cch - 1) / (32 / cch); }
// operands (16 bytes) of a slab of packed weights: [tile][step][part][lane]
template <typename S> __host__ __device__ inline size_t fused_slab_ops(int M, int kV, int cch) {
    return (size_t)fused_tiles(kV, cch) * fused_steps(M) * Parts<S>::NP * 64;
}
// operands of grad_output: [n][group][step][part][lane group][position]
template <typename S> inline size_t fused_gout_bytes(int N, int M, int G, size_t outV) {
    return (size_t)N * G * fused_steps(M) * Parts<S>::NP * 2 * outV * 16;
}

// Weights: lane (q, j) of step k in tile t holds the parts of W[m = 16 * k + 8 * q + e][channel = first + fused_row_channel(j)]
// [tap = t * 32 / CCH + fused_row_tap(j)], zero past M, the last tap and the segment.  A wavefront per tile and step.
template <int CCH, typename S>
__device__ inline void pack_fused_weight(const Params& P, const S* __restrict__ W, typename Parts<S>::Vec* __restrict__ Wq, unsigned block, unsigned blocks) {
    using PT = Parts<S>;
    constexpr int NP = PT::NP;
    const int steps = fused_steps(P.M), tiles = fused_tiles(P.kV, CCH);
    const unsigned per_slab = (unsigned)(tiles * steps), total = (unsigned)chunk_candidates<CCH>(P.cpg, P.Cg, P.C_in) * per_slab;      // wavefronts
    const int lane = threadIdx.x & 63, j = lane % 32;
    for (unsigned w = (unsigned)__builtin_amdgcn_readfirstlane(block * 4 + (threadIdx.x >> 6)); w < total; w += blocks * 4) {      // uniform for a wavefront
        const unsigned cand = w / per_slab, r = w - cand * per_slab;
        const int c0 = chunk_candidate<CCH>(P.cpg, P.Cg, (int)cand);
        const int g = c0 / P.Cg, dg = c0 / P.cpg, seg_b = max(dg * P.cpg, g * P.Cg), seg_e = min((dg + 1) * P.cpg, (g + 1) * P.Cg);
        if ((c0 - seg_b) % CCH) continue;
        const int t = (int)(r / (unsigned)steps), k = (int)r - t * steps;
        const int tap = t * (32 / CCH) + fused_row_tap<CCH>(j), c = c0 + fused_row_channel<CCH>(j), m0 = k * 16 + lane / 32 * 8;
        // (no load is masked: a masked one is waited for on its own)
        const S* src = W + ((size_t)g * P.M * P.Cg + (min(c, seg_e - 1) - g * P.Cg)) * P.kV + min(tap, P.kV - 1);
        S v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = src[(size_t)min(m0 + e, P.M - 1) * P.Cg * P.kV];
        typename PT::Vec part[NP];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            typename PT::Elem p[NP];
            PT::split1(m0 + e < P.M && tap < P.kV && c < seg_e ? v[e] : S(), p);
#pragma unroll
            for (int x = 0; x < NP; ++x) part[x][e] = p[x];
        }
        typename PT::Vec* dst = Wq + ((size_t)chunk_slot<CCH>(P.cpg, P.Cg, c0) * per_slab + r) * NP * 64 + lane;
#pragma unroll
        for (int x = 0; x < NP; ++x) dst[x * 64] = part[x];
    }
}

// grad_output in operand order, eight output channels of a position to a thread: both sides are contiguous over
// the positions.
template <typename S>
__device__ inline void split_grad_output(const Params& P, const S* __restrict__ gout, typename Parts<S>::Vec* __restrict__ gq, unsigned block, unsigned blocks) {
    using PT = Parts<S>;
    constexpr int NP = PT::NP;
    const int steps = fused_steps(P.M);
    const size_t total = (size_t)P.N * P.G * steps * 2 * P.outV;
    for (size_t i = (size_t)block * 256 + threadIdx.x; i < total; i += (size_t)blocks * 256) {
        unsigned pos;                                                   // of (n, group, step, lane group)
        int q, k;
        size_t ng;                                                      // n * G + g
        auto decode = [&](auto at) {
            const auto row = at / P.outV;
            pos = (unsigned)(at - row * P.outV);
            q = (int)(row & 1);
            ng = (row >> 1) / (unsigned)steps;
            k = (int)((row >> 1) - (decltype(at))ng * (unsigned)steps);
        };
        if (total <= ~0u) decode((unsigned)i);                          // (uniform; a 64-bit division is a hundred instructions)
        else decode(i);
        const int m0 = k * 16 + q * 8, left = P.M - m0;
        const S* src = gout + ng * P.M * P.outV + pos;
        S v[8];                                                         // (no load is masked: a masked one is waited for on its own)
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = src[(size_t)min(m0 + e, P.M - 1) * P.outV];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = e < left ? v[e] : S();
        typename PT::Vec part[NP];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            typename PT::Elem p[NP];
            PT::split1(v[e], p);
#pragma unroll
            for (int x = 0; x < NP; ++x) part[x][e] = p[x];
        }
        typename PT::Vec* dst = gq + (((ng * steps + k) * NP) * 2 + q) * (size_t)P.outV + pos;
#pragma unroll
        for (int x = 0; x < NP; ++x) dst[(size_t)x * 2 * P.outV] = part[x];
    }
}

constexpr int FUSED_WAVES = 16;
// tiles of a contraction: what 128 registers hold beside a tap slot.  (3-D: two of them, with half the loads of grad_output, cost 3 % on
// 64 channels at 27 taps.)
template <int ND, int CCH> __host__ __device__ inline constexpr int fused_pt() { return ND == 2 && CCH >= 8 ? 2 : 1; }
// LDS bytes per halo voxel: input cells (four float32 or eight 16-bit channels to 16 bytes) and the paired 32-bit sums
template <typename S> inline size_t fused_voxel_bytes(int cch) { return (size_t)((cch + HaloCell<S>::CH - 1) / HaloCell<S>::CH) * 16 + (size_t)cch * 4; }

// grad_input in octets, [n][channel / 8][voxel][8], where every chunk of channels is an octet or half of one: collected there, and brought to
// the layout of the tensor by octets_to_planes.  The float atomics of a flush go to memory by the line: 1.0e8 of them from halos of 9 x 15 x 15
// voxels take 545 us with the lanes along the rows of eight planes (14 voxels: 56 bytes), 283 in octets (448), 462 channels-last (32).
// Steps of 128 -> 128 in deformable groups of 32, stride 1 2 2, 2 x 16 x 112 x 112, in the tensor -> in octets: 4453 -> 4208 us (the kernel 2.40 -> 2.24 ms,
// 59 us for the tensor), of 64 -> 64, 4 x 16 x 56 x 56: 2398 -> 2358, in bfloat16 1618 -> 1606, whose flushes are a third as long beside the rest.
// put(index in the tensor, value), one thread per voxel of an octet.  last: the source is channels-last instead.
template <typename Put>
__device__ inline void octets_to_planes(const float* __restrict__ src, int N, int C, unsigned V, bool last, size_t first, size_t step, Put put) {
    typedef float F4 __attribute__((ext_vector_type(4)));
    const size_t items = (size_t)N * (unsigned)(C / 8) * V;
    for (size_t i = first; i < items; i += step) {
        const size_t row = items <= ~0u ? (size_t)((unsigned)i / V) : i / V;      // (uniform; a 64-bit division is a hundred instructions)
        const unsigned v = (unsigned)(i - row * V);
        const size_t n = row / (unsigned)(C / 8);
        const F4* from = reinterpret_cast<const F4*>(src + (last ? (n * V + v) * C + (row - n * (unsigned)(C / 8)) * 8 : i * 8));
        const F4 a = from[0], b = from[1];
#pragma unroll
        for (int e = 0; e < 8; ++e) put((row * 8 + e) * V + v, e < 4 ? a[e & 3] : b[e & 3]);
    }
}
// ADD: the tensor is added to.  *gate == gate_last: the source is channels-last.
template <bool ADD>
__global__ __launch_bounds__(256) void octets_to_planes_kernel(const float* __restrict__ src, float* __restrict__ dst, int N, int C, unsigned V,
                                                               const unsigned* __restrict__ gate, unsigned gate_last) {
    octets_to_planes(src, N, C, V, gate && *gate == gate_last, (size_t)blockIdx.x * 256 + threadIdx.x, (size_t)gridDim.x * 256, [&](size_t to, float v) {
        if (ADD) dst[to] += v;
        else dst[to] = v;
    });
}

// Dynamic LDS = hstride * fused_voxel_bytes(CCH).  Work items, csplit, whole and goff_atomic: as at backward_input_halo_kernel.
template <int ND, int CCH, int NPT, typename S>
__global__ __launch_bounds__(FUSED_WAVES * 64) void backward_fused_kernel(Params P, PlanSet alts, const unsigned* __restrict__ sel, const S* __restrict__ in,
                                                                          const S* __restrict__ off, const typename Parts<S>::Vec* __restrict__ Wq,
                                                                          const S* __restrict__ W, const S* __restrict__ gout,
                                                                          const typename Parts<S>::Vec* __restrict__ gq, const float* __restrict__ bounds,
                                                                          float* __restrict__ gin, float* __restrict__ goff, int csplit, unsigned whole,
                                                                          int goff_atomic, int octets) {
    touch_arguments<sizeof(Params) + sizeof(PlanSet) + 88>();
    HaloPlan H;
    if (!chosen_halo(P, alts, sel, H)) return;          // another launch runs the chosen plan
    using PS = Parts<S>;
    using Cells = LdsCell<float>;
    typedef typename PS::Vec Vec;
    typedef typename HaloCell<S>::Vec XCell;
    typedef unsigned long long Sum;
    constexpr int TN = 32, NC = 1 << ND, NP = PS::NP, CH = HaloCell<S>::CH;
    constexpr int PT = fused_pt<ND, CCH>(), NW = FUSED_WAVES, WGS = NW * 64, WPT = NW / NPT;      // wavefronts that share 32 positions
    constexpr int TP = 32 / CCH, NS = 16 / CCH;                         // taps and tap slots of a tile
    constexpr int XP = (CCH + CH - 1) / CH;                             // planes of input cells
    constexpr int CR = PT > 1 && NC > 4 ? 4 : NC;                        // corners read at a time
    constexpr int XR = 4;                                               // input cells of a thread in flight
    // The adds of a tap slot go ahead of what other wavefronts have to issue: 64 -> 64 channels, 3x3x3, 4 x 16 x 56 x 56, in bfloat16 a step 1630 -> 1595 us.
    // In float32, where the contraction has six times the instructions, 2371 -> 2364, at stride 1 2 2 4190 -> 4210, 2-D 877 -> 895.
    constexpr bool FIRST = ND == 3 && sizeof(S) == 2;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int hs = H.hstride;
    XCell* sIn = reinterpret_cast<XCell*>(smem_raw);                    // [XP][hs]
    Sum* sG = reinterpret_cast<Sum*>(sIn + (size_t)XP * hs);            // [CCH / 2][hs]
    __shared__ float sSq[WPT][NPT * TN], sMax[NW];
    __shared__ int sNonFinite[2];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % TN, q = lane / TN;
    const int pt = wave % NPT, wh = wave / NPT;         // position tile, share of its result tiles

    unsigned item;
    int cz = 0, cs = 1;
    if (blockIdx.x < whole) item = xcd_contiguous(blockIdx.x, whole);
    else {
        const unsigned r = xcd_contiguous(blockIdx.x - whole, gridDim.x - whole);
        cs = csplit;
        item = whole + r / (unsigned)cs;
        cz = (int)(r % (unsigned)cs);
    }
    const unsigned nt = (unsigned)P.N * (unsigned)P.tiles.d;
    const int dg = (int)(item / nt);
    goff_atomic = cs > 1 ? 1 : goff_atomic;

    TileGeo<ND> tg;
    tile_decode<ND>(P, H, item % nt, tg);
    const int n = tg.n;
    int ib[ND];
    unsigned pos;
    bool valid;
    {
        int o[ND];
        valid = tile_position<ND>(P, tg, pt * TN + j, o, pos);
#pragma unroll
        for (int a = 0; a < ND; ++a) ib[a] = o[a] * P.stride[slot<ND>(a)] - P.pad[slot<ND>(a)];
    }
    const unsigned row = (unsigned)H.hext[2], plane = ND == 3 ? (unsigned)(H.hext[1] * H.hext[2]) : 0u;
    const float inv2 = __builtin_amdgcn_rcpf((float)H.hext[2]), inv1 = __builtin_amdgcn_rcpf((float)H.hext[1]), invV = __builtin_amdgcn_rcpf((float)H.hvol);

    const int c_lo = dg * P.cpg, c_hi = c_lo + P.cpg;
    const S* off_dg = off + ((size_t)n * P.DG + dg) * P.kV * ND * P.outV;
    float* goff_dg = goff + ((size_t)n * P.DG + dg) * P.kV * ND * P.outV;
    const int steps = fused_steps(P.M), ntiles = (P.kV + TP - 1) / TP;
    const unsigned tap_lane = (unsigned)ND * P.outV;    // from a tap's offsets to the next tap's

    for (int i = threadIdx.x; i < CCH / 2 * hs; i += WGS) sG[i] = 0;
    if (threadIdx.x < 2) sNonFinite[threadIdx.x] = 0;
    bool first_chunk = true;                            // grad_offset without atomics: the first channel chunk stores, later ones add
    int chunk_no = 0, turn = 0;

    // The input cells of a chunk in two halves: their loads, up to XR cells of a thread, go out before the cells of the
    // chunk before are flushed (vector memory operations complete in order: behind the flush's atomics they would wait for
    // those), and reach the LDS afterwards.
    XCell xr[XR];
    // (a thread's number through an empty asm: what is derived from it is then worked out where it is used instead of
    // being kept in registers through the tap slots)
    auto here = [](unsigned v) { asm volatile("" : "+v"(v)); return v; };
    // Round u: a thread's voxel of the block u % xblocks of the halo, plane u / xblocks of the cells (uniform).
    const int xblocks = (H.hvol + WGS - 1) / WGS;
    auto load_cell = [&](const S* chan0, int nch, int u, XCell& cell) {
        const int pl = u / xblocks, vox = min((int)here(threadIdx.x) + (u - pl * xblocks) * WGS, H.hvol - 1);
        const unsigned at = halo_voxel<ND>(P, H, tg, vox, inv1, inv2);
        const unsigned byte = (at == ~0u ? 0u : at) * (unsigned)sizeof(S);
#pragma unroll
        for (int e = 0; e < CH; ++e)                                   // (no load is masked: a masked one is waited for on its own)
            if (e < CCH)
                cell[e] = HaloCell<S>::raw(*reinterpret_cast<const S*>(reinterpret_cast<const char*>(chan0 + (size_t)min(pl * CH + e, nch - 1) * P.inV) + byte));
    };
    auto store_cell = [&](int nch, int u, XCell cell) {
        const int pl = u / xblocks, vox = (int)here(threadIdx.x) + (u - pl * xblocks) * WGS;
        if (vox >= H.hvol) return;
        const bool there = halo_voxel<ND>(P, H, tg, vox, inv1, inv2) != ~0u;
        bool bad = false;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const bool real = e < CCH && pl * CH + e < nch && there;
            cell[e] = real ? cell[e] : (typename HaloCell<S>::V)0.f;
            bad = bad || !(fabsf((float)cell[e]) <= std::numeric_limits<float>::max());
        }
        sIn[(size_t)pl * hs + vox] = cell;
        if (bad) sNonFinite[turn] = 1;
    };
    auto load_x = [&](const S* chan0, int nch) {
        const int rounds = (nch + CH - 1) / CH * xblocks;
#pragma unroll
        for (int u = 0; u < XR; ++u) {
            load_cell(chan0, nch, min(u, rounds - 1), xr[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto store_x = [&](const S* chan0, int nch) {
        const int rounds = (nch + CH - 1) / CH * xblocks;
#pragma unroll
        for (int u = 0; u < XR; ++u)
            if (u < rounds) store_cell(nch, u, xr[u]);                 // (uniform)
        for (int u = XR; u < rounds; ++u) {
            XCell cell;
            load_cell(chan0, nch, u, cell);
            store_cell(nch, u, cell);
        }
    };

    // where the gradient of a voxel of this sample is collected
    auto gin_at = [&](int c, unsigned at) {
        return gin + (ND == 3 && octets ? ((size_t)n * P.C_in + (c & ~7)) * P.inV + (size_t)at * 8 + (c & 7) : ((size_t)n * P.C_in + c) * P.inV + at);
    };

    const int g_last = (c_hi - 1) / P.Cg;
#pragma unroll 1
    for (int g = c_lo / P.Cg; g <= g_last; ++g) {
        const int rb = max(c_lo, g * P.Cg), re = min(c_hi, (g + 1) * P.Cg);
        const int chunks = (re - rb + CCH - 1) / CCH, mine = (cz - chunk_no % cs + cs) % cs;      // this workgroup's: mine, mine + cs, ...
        chunk_no += chunks;
        if (mine >= chunks) continue;                                  // (uniform)
        auto chunk_input = [&](int cc0) { return in + ((size_t)n * P.C_in + cc0) * P.inV; };
        // (ahead of all else: the first latencies of a workgroup are a third of its time in layers of one chunk)
        load_x(chunk_input(rb + mine * CCH), min(CCH, re - (rb + mine * CCH)));
        // Scale of the fixed-point terms, from the norms of grad_output over the output channels: a term is at most the
        // largest column norm of W times the largest norm (Cauchy-Schwarz), a cell receives at most kV times the former times the
        // sum of the norms over the block.
        {
            const S* gm = gout + ((size_t)n * P.C_out + (size_t)g * P.M) * P.outV + pos;
            float ss = 0.f, am = 0.f;
            const int m0 = wh * 2 + q;
#pragma unroll 8
            for (int m = m0; m < P.M; m += 2 * WPT) {
                const float v = fabsf(Store<S>::ld(gm[(size_t)m * P.outV]));
                ss += v * v;
                am = v > am || v != v ? v : am;                        // (NaN stays: the comparison below then fails)
            }
            ss = valid ? ss : 0.f;
            am = valid ? am : 0.f;
            ss += __shfl_xor(ss, 32);
            unsigned ab = __float_as_uint(am);                         // (of the bit patterns, NaN is the largest)
#pragma unroll
            for (int sh = 1; sh < 64; sh <<= 1) ab = max(ab, (unsigned)__shfl_xor((int)ab, sh));
            __syncthreads();                                           // the last group's readers are done
            if (q == 0) sSq[wh][pt * TN + j] = ss;
            if (lane == 0) sMax[wave] = __uint_as_float(ab);
            __syncthreads();
        }
        float nsum = 0.f;
        unsigned nmaxb = 0u, gmaxb = 0u;
        for (int p = lane; p < NPT * TN; p += 64) {
            float ss = sSq[0][p];
#pragma unroll
            for (int w = 1; w < WPT; ++w) ss += sSq[w][p];
            const float norm = sqrtf(ss);
            nsum += norm;
            nmaxb = max(nmaxb, __float_as_uint(fabsf(norm)));
        }
#pragma unroll
        for (int sh = 1; sh < 64; sh <<= 1) {
            nsum += __shfl_xor(nsum, sh);
            nmaxb = max(nmaxb, (unsigned)__shfl_xor((int)nmaxb, sh));
        }
#pragma unroll
        for (int w = 0; w < NW; ++w) gmaxb = max(gmaxb, __float_as_uint(sMax[w]));
        const float gmax = __uint_as_float(gmaxb), wcol = weight_bound(bounds, 1), wmax = weight_bound(bounds, 0);
        const float bound = 1.001f * wcol * __uint_as_float(nmaxb);    // (0.1 % for the rounding of the norms and of the contraction)
        const float bound_cell = 1.001f * wcol * (float)P.kV * nsum;
        // Without a finite bound, where the squares of a tiny grad_output underflow, or where the scale would leave the range of a float,
        // the workgroup scatters through global memory (false for NaN).
        const bool cells_ok = bound < 3.0e38f && bound_cell < 3.0e38f && !(gmax > 0.f && gmax < 1e-18f) && !(gmax > 0.f && wcol > 0.f && bound < 1e-30f);
        // operands that bfloat16 parts do not hold: the contraction on the float32 instructions
        const bool exact_all = sizeof(S) == 4 && !(cells_ok && gmax < 0x1p126f && wmax < 0x1p126f && !(wmax > 0.f && wmax < 1e-18f));
        float scale = 1.f;
        if (bound > 0.f && cells_ok) {
            // a single term stays below 2^22 (the float conversion of add2), all that a cell can receive below 2^31
            // (half a unit of rounding each for at most NPT * 32 * kV terms fits the one per cent of slack)
            const double s_term = 4194304.0 / (double)bound;
            const double s_cell = bound_cell > 0.f ? 2147483648.0 / (double)bound_cell : s_term;
            scale = (float)(0.99 * (s_term < s_cell ? s_term : s_cell));
        }
        scale = __uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)__float_as_uint(scale)));
        const double inv_scale = 1.0 / (double)scale;
        const Vec* gqg = gq + ((size_t)n * P.G + g) * steps * NP * 2 * P.outV;

        const size_t wslab = (size_t)ntiles * steps * NP * 64;
        auto chunk_weights = [&](int cc0) { return Wq + (size_t)chunk_slot<CCH>(P.cpg, P.Cg, cc0) * wslab; };

        Mma<float>::Acc acc[PT];
        float ofs[ND], prev[ND];
#pragma unroll
        for (int a = 0; a < ND; ++a) prev[a] = 0.f;
        // offsets of a tap slot, and what the earlier chunks have written to its grad_offset (rmw)
        auto load_slot = [&](int tap0, bool rmw) {                     // tap0: lane group 0's tap (uniform)
            const S* ob = off_dg + (size_t)tap0 * ND * P.outV;
            const unsigned lo = here((q && tap0 + 1 < P.kV ? tap_lane : 0u) + pos);
#pragma unroll
            for (int a = 0; a < ND; ++a) ofs[a] = Store<S>::ld((ob + (size_t)a * P.outV)[lo]);
            if (rmw) {
                const float* gb = goff_dg + (size_t)tap0 * ND * P.outV;
#pragma unroll
                for (int a = 0; a < ND; ++a) prev[a] = (gb + (size_t)a * P.outV)[lo];
            }
        };
        // The contraction of the tiles tb + wh + WPT * p (p < PT) of a chunk.
        auto contract = [&](int cc0, int tb) {
            const int t0 = tb + wh, left = t0 < ntiles ? (ntiles - t0 + WPT - 1) / WPT : 0;
            const Vec* wq = chunk_weights(cc0);
            const Vec* bp = gqg;
            const unsigned b_lane = here((unsigned)q * P.outV + pos), a_lane = here(lane);
#pragma unroll
            for (int p = 0; p < PT; ++p) acc[p] = acc_zero<float>();
            if (left > 0) {
                const Vec* wp = wq + (size_t)t0 * steps * NP * 64;
                for (int k = 0; k < steps; ++k) {
                    Vec b8[NP], a8[PT][NP];
#pragma unroll
                    for (int x = 0; x < NP; ++x) b8[x] = (bp + (size_t)x * 2 * P.outV)[b_lane];
#pragma unroll
                    for (int p = 0; p < PT; ++p)
                        if (p < left) {
#pragma unroll
                            for (int x = 0; x < NP; ++x) a8[p][x] = (wp + (size_t)p * WPT * steps * NP * 64 + x * 64)[a_lane];
                        }
#pragma unroll
                    for (int p = 0; p < PT; ++p)
                        if (p < left) mma_parts<S, 1>(&a8[p], b8, &acc[p]);
                    wp += NP * 64;
                    bp += (size_t)NP * 2 * P.outV;
                }
            }
            if constexpr (sizeof(S) == 4) {
                // results that parts may have cost bits (see dcn_forward_split.h), and operands without parts
                unsigned least = ~0u;
#pragma unroll
                for (int p = 0; p < PT; ++p)
#pragma unroll
                    for (int r = 0; r < 16; ++r) least = min(least, (__float_as_uint(acc[p][r]) << 1) - 1u);
                if (__builtin_expect(exact_all || __any(valid && least < (__float_as_uint(0x1p-80f) << 1) - 1u), 0)) {
#pragma unroll
                    for (int p = 0; p < PT; ++p)
                        if (p < left) {
                            const int tap = (t0 + p * WPT) * TP + fused_row_tap<CCH>(j), c = cc0 + fused_row_channel<CCH>(j);
                            const bool real = tap < P.kV && c < re;
                            acc[p] = acc_zero<float>();
#pragma unroll 1
                            for (int m0 = 0; m0 < P.M; m0 += 2) {
                                const int m = min(m0 + q, P.M - 1);
                                float a = 0.f, b = 0.f;
                                if (real && m0 + q < P.M) a = Store<S>::ld(W[(((size_t)g * P.M + m) * P.Cg + (c - g * P.Cg)) * P.kV + tap]);
                                if (m0 + q < P.M) b = Store<S>::ld(gout[((size_t)n * P.C_out + (size_t)g * P.M + m) * P.outV + pos]);
                                acc[p] = Mma<float>::mma(a, b, acc[p]);
                            }
                        }
                }
            }
        };
        contract(rb + mine * CCH, 0);
        store_x(chunk_input(rb + mine * CCH), min(CCH, re - (rb + mine * CCH)));
        __syncthreads();
        for (int ci = mine; ci < chunks; ci += cs) {
            const int cc0 = rb + ci * CCH, nch = min(CCH, re - cc0);
            // Non-finite input values in this halo: samples in the collapse zones (p <= 0 or p >= size - 1 on some axis) take
            // the far path, which follows the reference's corner rule; the branch-free sampler reads the cell next to a
            // collapsed corner with weight 0, and 0 * inf would be NaN where the reference never touches that voxel
            // (deform3d/lib/deform_conv3d_cuda_kernel.cu:24-26).
            const bool rim_far = sNonFinite[turn] != 0;
            turn ^= 1;
            if (threadIdx.x == 0) sNonFinite[turn] = 0;                // (set again behind the barrier at the end of this chunk)
            const bool rmw_prev = ND == 3 && !goff_atomic && !first_chunk;

            for (int tb = 0; tb < ntiles; tb += WPT * PT) {
                const int t0 = tb + wh, left = t0 < ntiles ? (ntiles - t0 + WPT - 1) / WPT : 0;
                if (left > 0) load_slot(t0 * TP, rmw_prev);
                if (tb > 0) contract(cc0, tb);
#pragma unroll
                for (int p = 0; p < PT; ++p) {
                    if (p >= left) break;                              // (uniform)
                    const int tile_tap = (t0 + p * WPT) * TP;
                    int k0[ND];
                    decode_tap<ND>(P, tile_tap, k0);
#pragma unroll
                    for (int ts = 0; ts < NS; ++ts) {
                        const int tap0 = tile_tap + 2 * ts;            // lane group 0's tap
                        if (tap0 >= P.kV) break;                       // (uniform)
                        const int tap = tap0 + q;
                        int k1[ND];
#pragma unroll
                        for (int a = 0; a < ND; ++a) k1[a] = k0[a];
                        next_tap<ND>(P, k1);
                        float gv[CCH];
#pragma unroll
                        for (int e = 0; e < CCH; ++e) gv[e] = acc[p][ts * CCH + e];

                        // Geometry, following the reference sampler (deform3d/lib/deform_conv3d_cuda_kernel.cu:21-26,40-45,123-124)
                        // in a branch-free form, see split_geometry.
                        const bool slot_ok = valid && tap < P.kV;
                        bool inside = slot_ok, inhalo = cells_ok, intr[ND];
                        float pq[ND], f[ND], prv[ND];
                        int u[ND];
#pragma unroll
                        for (int a = 0; a < ND; ++a) {
                            const int sa = slot<ND>(a);
                            const float top = (float)(P.in[sa] - 1);
                            const int kd = k0[a] * P.dil[sa];
                            int dk = k1[a] * P.dil[sa] - kd;
                            asm volatile("" : "+s"(dk));               // (scalar arithmetic)
                            const float pa = (float)(__mul24(q, dk) + ib[a] + kd) + ofs[a];
                            const float pc = __builtin_amdgcn_fmed3f(pa, 0.f, top);
                            const float fl = floorf(pc);
                            pq[a] = pa;
                            f[a] = pc - fl;
                            inside = inside && fabsf(pa - pc) < 1.f;   // -1 < p < size, false for NaN
                            intr[a] = pa > 0.f && pa < top;            // strictly between the collapse zones: the axis has a slope
                            u[a] = (int)fl - tg.hb[a];
                            inhalo = inhalo && (unsigned)u[a] < (unsigned)(H.hext[sa] - 1);
                            prv[a] = prev[a];
                        }
                        if (rim_far) {
#pragma unroll
                            for (int a = 0; a < ND; ++a) inhalo = inhalo && intr[a];
                        }
                        const bool near = inside && inhalo, far = inside && !inhalo;
                        unsigned base;
                        if constexpr (ND == 3) base = (unsigned)(__mul24(__mul24(u[0], H.hext[1]) + u[1], H.hext[2]) + u[2]);
                        else base = (unsigned)(__mul24(u[0], H.hext[2]) + u[1]);
                        base = near ? base : 0u;                       // lanes without a sample in the halo read cell 0 and add nothing
                        // the next slot of this round
                        if (ts + 1 < NS && tap0 + 2 < P.kV) load_slot(tap0 + 2, rmw_prev);
                        else if (p + 1 < PT && p + 1 < left) load_slot((t0 + (p + 1) * WPT) * TP, rmw_prev);

                        // Corner values weighted by the grad columns and summed over the channels: the derivative of the sample
                        // is linear in them.  Every lane reads, outside any branch (corner reads still pending at a branch
                        // that skips their use would make the compiler wait for the whole LDS queue, adds included).
                        float v[NC];
#pragma unroll
                        for (int i = 0; i < NC; ++i) v[i] = 0.f;
#pragma unroll
                        for (int x = 0; x < XP; ++x) {
                            if (x * CH >= nch) break;                  // (uniform)
                            const XCell* xp = sIn + base + (size_t)x * hs;
#pragma unroll
                            for (int i0 = 0; i0 < NC; i0 += CR) {      // (CR corners at a time, for the registers)
                                XCell c[CR];
#pragma unroll
                                for (int i = 0; i < CR; ++i) c[i] = xp[((i0 + i) >> 2) * plane + (((i0 + i) >> 1) & 1) * row + ((i0 + i) & 1)];
#pragma unroll
                                for (int i = 0; i < CR; ++i)
#pragma unroll
                                    for (int e = 0; e < CH && x * CH + e < CCH; ++e) v[i0 + i] += gv[x * CH + e] * (float)c[i][e];
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        }
                        float ga[ND];
                        if constexpr (ND == 3) {
                            const float fl = f[0], gl = 1.f - fl, fh = f[1], gh = 1.f - fh, fw = f[2], gw = 1.f - fw;
                            const float c00 = v[0] * gw + v[1] * fw, c01 = v[2] * gw + v[3] * fw;
                            const float c10 = v[4] * gw + v[5] * fw, c11 = v[6] * gw + v[7] * fw;
                            const float dl = (c10 - c00) * gh + (c11 - c01) * fh;
                            const float dh = (c01 - c00) * gl + (c11 - c10) * fl;
                            const float dw = ((v[1] - v[0]) * gh + (v[3] - v[2]) * fh) * gl + ((v[5] - v[4]) * gh + (v[7] - v[6]) * fh) * fl;
                            ga[0] = near && intr[0] ? dl : 0.f;
                            ga[1] = near && intr[1] ? dh : 0.f;
                            ga[2] = near && intr[2] ? dw : 0.f;
                        } else {
                            const float fh = f[0], gh = 1.f - fh, fw = f[1], gw = 1.f - fw;
                            const float dh = (v[2] - v[0]) * gw + (v[3] - v[1]) * fw;
                            const float dw = (v[1] - v[0]) * gh + (v[3] - v[2]) * fh;
                            ga[0] = near && intr[0] ? dh : 0.f;
                            ga[1] = near && intr[1] ? dw : 0.f;
                        }
                        if (near) {
                            float cw[NC];                              // corner weights (the reference's order w_l * w_h * w_w), scaled
                            if constexpr (ND == 3) {
                                const float fl = f[0] * scale, gl = (1.f - f[0]) * scale, fh = f[1], gh = 1.f - fh, fw = f[2], gw = 1.f - fw;
                                const float a00 = gl * gh, a01 = gl * fh, a10 = fl * gh, a11 = fl * fh;
                                cw[0] = a00 * gw; cw[1] = a00 * fw; cw[2] = a01 * gw; cw[3] = a01 * fw;
                                cw[4] = a10 * gw; cw[5] = a10 * fw; cw[6] = a11 * gw; cw[7] = a11 * fw;
                            } else {
                                const float fh = f[0] * scale, gh = (1.f - f[0]) * scale, fw = f[1], gw = 1.f - fw;
                                cw[0] = gh * gw; cw[1] = gh * fw; cw[2] = fh * gw; cw[3] = fh * fw;
                            }
                            Sum* cp = sG + base;
                            if constexpr (FIRST) __builtin_amdgcn_s_setprio(1);
#pragma unroll
                            for (int e = 0; e < CCH; e += 2) {
#pragma unroll
                                for (int i = 0; i < NC; ++i)
                                    Cells::add2(cp + (i >> 2) * plane + ((i >> 1) & 1) * row + (i & 1), cw[i], gv[e], gv[e + 1]);
                                cp += hs;
                            }
                            if constexpr (FIRST) __builtin_amdgcn_s_setprio(0);
                        }
                        if constexpr (ND == 3) {
                            // out-of-range samples of the 3-D operator: -|gcol| per axis with p <= -1, +|gcol| with p >= the LENGTH extent
                            // (h and w are compared with it too), summed over the channels
                            // (deform3d/lib/deform_conv3d_cuda_kernel.cu:470-481).  Selected, not multiplied: 0 * inf would be NaN, and
                            // is in the columns past the chunk's channels, whose weights are zeros
                            const bool oor = slot_ok && !inside && !P.oob_zero;
                            if (__any(oor)) {
                                float asum = 0.f;
                                int real = nch;
                                asm volatile("" : "+s"(real));         // (compared here: hoisted, the comparisons spill scalar registers)
#pragma unroll
                                for (int e = 0; e < CCH; ++e) asum += e < real ? fabsf(gv[e]) : 0.f;
                                if (oor) {
#pragma unroll
                                    for (int a = 0; a < ND; ++a) ga[a] = pq[a] <= -1.f ? -asum : (pq[a] >= (float)P.in[0] ? asum : 0.f);
                                }
                            }
                        }
                        if (__builtin_expect(__any(far), 0)) {         // samples that reach past the halo: global memory
                            // 3-D and 16-bit storage: the samples one after the other, a lane for each of a sample's (corner, channel) pairs, one round trip
                            // to memory each.  A loop over the channels with the samples in their lanes waits for as many round trips as there are
                            // channels however few the samples, and its spills cost the tap slots (us of a call, that loop -> this: 64 -> 64, 3x3x3, 200 704
                            // positions, offsets U[-1.5, 1.5] 1311 -> 1272, N(0, 0.7) 1865 -> 1284, at margin 2 N(0, 1) 2932 -> 1682 and U[-3, 3] 5737 -> 3902; in
                            // bfloat16, 50 176 positions, U[-6, 6] 9591 -> 5783).  float32 in 2-D, where wide halos are cheap and far samples rare: the loop
                            // (steps of 512 -> 512 in two groups 328 us, 331 with this).
                            if constexpr (ND == 2 && sizeof(S) == 4) {
                                TapGeo<float, ND> t;                       // the reference's corner rule on the same coordinate
                                t.inside = far;
#pragma unroll
                                for (int a = 0; a < ND; ++a) {
                                    float pa = pq[a];
                                    asm volatile("" : "+v"(pa));           // (worked out here, not hoisted into the common path)
                                    const int l = far ? (int)pa : 0;
                                    t.p[a] = pa;
                                    t.lo[a] = l;
                                    t.hi[a] = (pa >= (float)(P.in[slot<ND>(a)] - 1) || pa <= 0.f) ? l : l + 1;
                                    t.f[a] = pa - (float)l;
                                }
                                tap_corner_idx<float, ND>(P, t);
#pragma unroll 1
                                for (int e = 0; e < nch; ++e) {
                                    float g1 = 0.f;
#pragma unroll
                                    for (int x = 0; x < CCH; ++x) g1 = x == e ? gv[x] : g1;
                                    const size_t chan = ((size_t)n * P.C_in + cc0 + e) * P.inV;
                                    if (far) {
                                        const S* ic = in + chan;
                                        float vv[NC];
#pragma unroll
                                        for (int i = 0; i < NC; ++i) vv[i] = g1 * Store<S>::ld(ic[t.idx[i]]);
                                        const float fh = t.f[0], gh = 1.f - fh, fw = t.f[1], gw = 1.f - fw;
                                        const float cw[4] = {gh * gw, gh * fw, fh * gw, fh * fw};
#pragma unroll
                                        for (int i = 0; i < NC; ++i) atomic_add(gin_at(cc0 + e, t.idx[i]), cw[i] * g1);
                                        ga[0] += (vv[2] - vv[0]) * gw + (vv[3] - vv[1]) * fw;
                                        ga[1] += (vv[1] - vv[0]) * gh + (vv[3] - vv[2]) * fh;
                                    }
                                }
                            } else {
                                unsigned long long todo = __ballot(far);
#pragma unroll 1
                                while (todo) {                         // (a bit less each time)
                                    const int src = __builtin_ctzll(todo), me = (int)here((unsigned)lane), i = me % NC, e = me / NC;
                                    todo &= todo - 1;
                                    auto from = [&](float v) { return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(v), src)); };
                                    float g1 = 0.f, wa[ND], d[ND];
#pragma unroll
                                    for (int x = 0; x < CCH; ++x) g1 = x == e ? from(gv[x]) : g1;
                                    unsigned at = 0;
#pragma unroll
                                    for (int a = 0; a < ND; ++a) {     // the reference's corner rule on the same coordinate
                                        const int size = P.in[slot<ND>(a)];
                                        const float pa = from(pq[a]);
                                        const int l = (int)pa, up = (i >> (ND - 1 - a)) & 1;
                                        at = at * (unsigned)size + (unsigned)(l + (up && !(pa >= (float)(size - 1) || pa <= 0.f) ? 1 : 0));
                                        wa[a] = up ? pa - (float)l : 1.f - (pa - (float)l);
                                        d[a] = 0.f;
                                    }
                                    if (e < nch) {
                                        const float v = g1 * Store<S>::ld(in[((size_t)n * P.C_in + cc0 + e) * P.inV + at]);
                                        float cw = wa[0];
#pragma unroll
                                        for (int a = 1; a < ND; ++a) cw *= wa[a];
                                        atomic_add(gin_at(cc0 + e, at), cw * g1);
#pragma unroll
                                        for (int a = 0; a < ND; ++a) {
                                            d[a] = (i >> (ND - 1 - a)) & 1 ? v : -v;
#pragma unroll
                                            for (int b = 0; b < ND; ++b)
                                                if (b != a) d[a] *= wa[b];
                                        }
                                    }
#pragma unroll
                                    for (int a = 0; a < ND; ++a) {
                                        d[a] = group_sum(d[a]);        // (its holders: the last lanes of either half)
                                        const float sum = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(d[a]), 31)) +
                                                          __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(d[a]), 63));
                                        ga[a] += me == src ? sum : 0.f;
                                    }
                                }
                            }
                        }
                        if (slot_ok) {
                            float* gp = goff_dg + (size_t)tap0 * ND * P.outV;
                            const unsigned lo = here((q ? tap_lane : 0u) + pos);
#pragma unroll
                            for (int a = 0; a < ND; ++a) {
                                float* p1 = (gp + (size_t)a * P.outV) + lo;
                                if (goff_atomic) { if (ga[a] != 0.f) atomic_add(p1, ga[a]); }
                                else if (ND == 3 || first_chunk) *p1 = rmw_prev ? ga[a] + prv[a] : ga[a];
                                else *p1 += ga[a];
                            }
                        }
                        next_tap<ND>(P, k1);
#pragma unroll
                        for (int a = 0; a < ND; ++a) k0[a] = k1[a];
                        __builtin_amdgcn_sched_barrier(0);             // one tap slot at a time: keeps the live register set small
                    }
                }
            }
            first_chunk = false;
            // the next chunk's first contraction and input loads go out before this one's sums
            const int cn = cc0 + cs * CCH, nchn = min(CCH, re - cn);
            const bool more = ci + cs < chunks;                        // (uniform)
            if (more) {
                contract(cn, 0);
                load_x(chunk_input(cn), nchn);
            }
            __syncthreads();                                           // all LDS adds of this chunk have landed
            constexpr int FE = CCH < 8 ? CCH : 8, FP = FE / 2;         // channels, cell planes flushed together
            if (ND == 3 && octets) {
                // 64 voxels to a wavefront: each works one out, then FE lanes share a voxel, whose sums go to neighbouring addresses
                const unsigned l = here((unsigned)lane), e = l % FE;
                float* const ge = gin + ((size_t)n * P.C_in + (cc0 & ~7)) * P.inV + (cc0 & 7) + e;
                for (int v0 = wave * 64; v0 < H.hvol; v0 += WGS) {
                    const int vox = v0 + (int)l;
                    const unsigned at = vox < H.hvol ? halo_voxel<ND>(P, H, tg, vox, inv1, inv2) : ~0u;
                    Sum* const cp = sG + (size_t)(e / 2) * hs;
                    int from[FE];
                    unsigned to[FE];
                    Sum cell[FE];
#pragma unroll
                    for (int u = 0; u < FE; ++u) {
                        to[u] = (unsigned)__shfl((int)at, u * (64 / FE) + (int)(l / FE));
                        from[u] = min(v0 + u * (64 / FE) + (int)(l / FE), H.hvol - 1);
                        cell[u] = cp[from[u]];
                    }
                    // Both lanes of a cell have read it before each clears its half, through a type that may stand for the cell's: without either the
                    // order of the two is the compiler's.  (The whole cell cleared, by both lanes or one: bfloat16 steps 1603 -> 1618 us.)
                    typedef unsigned __attribute__((may_alias)) Half;
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
                    __builtin_amdgcn_sched_barrier(0);                 // all of them on their way
#pragma unroll
                    for (int u = 0; u < FE; ++u)
                        if (to[u] != ~0u) {                            // (a cell outside the volume holds zero)
                            reinterpret_cast<Half*>(cp + from[u])[e & 1] = 0;
                            const float v = Cells::value_of_pair(cell[u], e & 1, inv_scale);
                            if (v != 0.f) atomic_add(ge + (size_t)to[u] * 8, v);
                        }
                }
            } else {
                const int pairs = (nch + 1) / 2, cells = (pairs + FP - 1) / FP * H.hvol;
                for (int it = (int)here(threadIdx.x); it < cells; it += WGS) {
                    const int pg = CCH > 8 ? (int)(((float)it + 0.5f) * invV) : 0, vox = it - __mul24(pg, H.hvol);
                    const unsigned at = halo_voxel<ND>(P, H, tg, vox, inv1, inv2);
                    float* gp = gin + ((size_t)n * P.C_in + cc0 + pg * 8) * P.inV + (at == ~0u ? 0u : at);
                    Sum* cp = sG + (size_t)(pg * 4) * hs + vox;
                    Sum cell[FP];
#pragma unroll
                    for (int x = 0; x < FP; ++x) cell[x] = cp[(size_t)x * hs];
#pragma unroll
                    for (int x = 0; x < FP; ++x) cp[(size_t)x * hs] = 0;
                    if (at == ~0u) continue;                           // (a cell outside the volume holds zero)
#pragma unroll
                    for (int x = 0; x < FP; ++x) {                     // (planes past the chunk's channels hold zeros)
                        float v0, v1;
                        Cells::value2(cell[x], inv_scale, v0, v1);
                        if (v0 != 0.f) atomic_add(gp, v0);
                        if (pg * 8 + x * 2 + 1 < nch && v1 != 0.f) atomic_add(gp + P.inV, v1);
                        gp += 2 * (size_t)P.inV;
                    }
                }
            }
            if (more) {
                store_x(chunk_input(cn), nchn);
                __syncthreads();
            }
        }
    }
}

}  // namespace dcn
