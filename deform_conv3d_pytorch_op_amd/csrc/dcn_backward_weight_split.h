// Backward pass to the weight of the float32 and 16-bit operators, for layers of more than 32 output channels to a group or few channels
// to a segment (split_plan).
//
//   gW[g*M+m][cl][tap] += sum_{n,pos} grad_output[n][g*M+m][pos] * sample(in[n][g*Cg+cl], tap, pos)
//
// replaces the second deformable_im2col + Sgemm(beta=1) of deform3d/lib/deform_conv3d_cuda.cpp:283-320.
//
// The reduction runs over positions.  A wavefront samples 32 channels of one tap (16-bit storage: 64, two to a lane; few channels: LW lanes
// to each of 32 / LW taps): lane
// (j, q) takes channel c0 + j at eight consecutive positions of a step of 16 -- the input is channels-last, so a corner is one
// coalesced 128-byte read of the lane group -- and those eight samples are the lane's operand of v_mfma_f32_32x32x16_bf16 / _f16
// as they stand: three bfloat16 parts or one of the storage format (dcn_forward_split.h).  The other operand, the rows of
// grad_output, comes from the preparing launch in operand order (prep_rows); the four wavefronts of a workgroup work taps or channel tiles of their own on the same positions and share it
// through LDS, two steps of it in turn.  The geometry of a slab of 32 positions is worked out once by the position-owning
// lanes and handed to the channel lanes through a wavefront-private record: byte offset of the low corner and the corner
// weights.  The low corner is at most size - 2, so that the other corners lie at fixed strides (scalar bases of their own, one
// address per lane and position for all of them) and a corner past the rim is never read.
// An accumulator stays in registers for the whole run of a wavefront, which writes one partial tile;
// reduce_weight_partials_kernel sums the splits (deterministic, no atomics).  Results that are not finite or too small for the
// parts are formed once more from the values themselves.
// The instruction cuts what lies below the last places of a product off towards minus infinity, and a chain of hundreds of
// steps adds that up: the products of a step are summed from zero and then added, and every second split samples with its sign
// turned round and turns its tile back.  Error of grad_weight against float64 (2-norm; 64 -> 64, 3x3x3, 4 x 16 x 56 x 56, whose rounded
// coordinates make 2.0e-6 of it; 64 -> 64, 3x3, no offsets): float32 instructions 2.00e-6 and 1.84e-7, one chain 2.39e-6 and
// 2.51e-7, with sums of a step 2.15e-6 and 3.66e-7, with the signs as well 2.00e-6 and 1.51e-7.
//
// What bounds it: the corner reads.  64 -> 64 channels, 3x3x3, 4 x 16 x 56 x 56 positions: 12.2 GB through the vector caches,
// whose data return is busy 96 % of the time (8.5 GB from L2), the matrix units 20 %, the vector units 40 %.  backward_weight_kernel
// with the float32 instructions kept the matrix units busy half of the time and read grad_output once per wavefront: with rows
// straight from L2 this kernel was no faster in 3-D (678 us against 633) and 13 % faster in 2-D.  us of the kernel alone, that one -> this one: 256 -> 256,
// 3x3, 8 x 56 x 56: 332 -> 240; 512 -> 512 in two groups, 3x3, 4 x 28 x 28: 105 -> 80; 128 -> 128, 3x3x3, 2 x 16 x 56 x 56
// (stride 2): 1022 -> 860; 64 -> 64 as above: 633 -> 600; 64 -> 64, 3x3, no offsets, 25 088 positions: 33 -> 25.
// The preparing launch pays 2 to 20 us of it back (three halves of the bytes of a channels-last copy).
// float32 layers of more than 128 output channels to a group, where they pay (eight_tiles_pay): eight row tiles, so that 256 of them share the corner reads
// of a sample, at two wavefronts per SIMD instead of three: 256 -> 256 as above 228 -> 208 (steps of the layer 900 -> 889 us).  In 16-bit
// storage a lane holds two column tiles and eight row tiles leave one wavefront per SIMD: steps of 256 -> 256 in binary16 497 -> 514 us, so it keeps four.
// Where every lane's channels are aligned to it (QUAD), eight lanes read 16 bytes of a corner each and the wavefront eight positions at a time: a
// quarter of the load instructions -- of a line or a half to a lane group, one that hits the L1 takes 7.5 ns a CU for 1 KB, of 4 bytes to a lane 2.9 for 256
// bytes -- and of the records, and the weighted sums change places with the positions (swap_lanes_registers) before the
// contraction.  2-D and 16-bit storage: us of the kernel alone, 4 bytes -> 16: 256 -> 256 in binary16 118 -> 95 (step 466 -> 433),
// in float32 208 -> 193, without offsets 26.7 -> 23.7, 64 -> 64 in 3-D in bfloat16 333 -> 289 (step 1752 -> 1717).  Not float32 in 3-D, where the lines of eight positions with eight corners each, of every wavefront, turn the L1 over before their
// neighbours come back to them: steps of 64 -> 64 2478 -> 2598 us, of 128 -> 128 4525 -> 5058.
// 16-bit storage, against backward_weight16_kernel, which samples once for every 64 output channels: 256 -> 256 in float16 150 -> 116,
// 64 -> 64 in 3-D in bfloat16 361 -> 326.
#pragma once
#include <cmath>
#include "dcn_forward_split.h"

namespace dcn {

constexpr unsigned ROW_SLAB = 32;                       // positions of a slab: two steps
__host__ __device__ inline unsigned row_steps(unsigned V) { return (V + ROW_SLAB - 1) / ROW_SLAB * 2; }
// grad_output in operand order: [n][octet of positions][part][output channel], 16 bytes (eight positions) each, zero past the volume
template <typename S> inline size_t row_operand_bytes(int N, int C_out, size_t V) { return (size_t)N * row_steps((unsigned)V) * Parts<S>::NP * 2 * C_out * 16; }
// channels to a lane (16-bit storage: pairs, two column tiles)
template <typename S> __host__ __device__ constexpr int lane_channels() { return 4 / (int)sizeof(S); }

// wavefronts to a SIMD
template <typename S> __host__ __device__ constexpr int split_waves(int MT) { return MT == 8 ? 2 : (MT == 4 ? 3 : 4) - (sizeof(S) == 2); }

// channel u of what a lane reads of a corner
template <typename S> __device__ inline float channel_of(float v, int) { return v; }
template <typename S> __device__ inline float channel_of(unsigned v, int u) {
    if constexpr (std::is_same<S, Bf16>::value) return __uint_as_float(u ? v & 0xffff0000u : v << 16);
    else return (float)__builtin_bit_cast(_Float16, (unsigned short)(u ? v >> 16 : v));
}
typedef unsigned Quad __attribute__((ext_vector_type(4)));
template <typename S> __device__ inline float channel_of(const Quad& v, int u) {
    if constexpr (sizeof(S) == 4) return __uint_as_float(v[u]);
    else return channel_of<S>(v[u / 2], u % 2);
}

// Where bit `lane bit 4` of a lane's number and one of the two registers trade places, then bit 3: registers v[k1 * 2 + k0] of lanes (.., p1, p0, ...)
// become v[p1 * 2 + p0] of lanes (.., k1, k0, ...).
__device__ inline void swap_lanes_registers(float v[4]) {
    auto bits = [](float x) { return __float_as_uint(x); };
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const auto r = __builtin_amdgcn_permlane16_swap(bits(v[k]), bits(v[2 + k]), false, false);      // odd rows of the first with even rows of the second
        v[k] = __uint_as_float(r[0]);
        v[2 + k] = __uint_as_float(r[1]);
    }
#pragma unroll
    for (int k = 0; k < 4; k += 2) {                    // row_ror:8, written to the upper eight lanes of a row or to the lower
        const unsigned a = bits(v[k]), b = bits(v[k + 1]);
        v[k] = __uint_as_float(__builtin_amdgcn_update_dpp(a, b, 0x128, 0xF, 0xC, false));
        v[k + 1] = __uint_as_float(__builtin_amdgcn_update_dpp(b, a, 0x128, 0xF, 0x3, false));
    }
}

// MT row tiles to a workgroup.  LW lanes to a tap: an item is 32 / LW taps of LW channels (pairs).  PLAIN: a plain convolution (off is null): samples at integer coordinates are their low corner alone.
// Grid: igroups * mchunks * G * nsplit workgroups.  The items of a convolution group: taps of a channel tile, taps fastest.
// QUAD: 16 bytes of a corner to a lane -- see the top of the file and split_quad; channels and segments in multiples of four (16-bit storage: eight).
template <int ND, int MT, int LW, typename S, bool QUAD, bool PLAIN = false>
__global__ __launch_bounds__(WG, split_waves<S>(MT)) void backward_weight_split_kernel(Params P, const S* __restrict__ in_cl, const S* __restrict__ off,
                                                                                         const S* __restrict__ gout,
                                                                                         const typename Parts<S>::Vec* __restrict__ rows,
                                                                                         float* __restrict__ partial, unsigned igroups) {
    typedef float T;
    using MM = Mma<float>;
    using PT = Parts<S>;
    typedef typename PT::Vec Vec;
    constexpr int CT = lane_channels<S>(), TC = LW * CT;        // channels of a lane, of a tap
    constexpr int TP = 32 / LW, GT = TP > 1 ? TP / 2 : 1;       // taps of an item, of a lane that works out geometry
    constexpr int TN = 32, NP = PT::NP, NC = 1 << ND, NR = PLAIN ? 1 : NC;     // corners, corners read
    touch_arguments<sizeof(Params) + 40>();
    __shared__ unsigned sIdx[WAVES][TP][TN];                      // byte offset of the low corner's channel 0 inside the sample
    __shared__ __align__(16) T sCw[WAVES][TP][TN][NR];            // weight of each corner, 0 where there is no sample
    __shared__ __align__(16) unsigned char sRow[2][MT * NP * 1024];        // rows of a step of grad_output: [part][q][row]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane % TN, q = lane / TN;

    // XCD-contiguous order with the items fastest: the workgroups that gather around the same positions share an L2
    unsigned wg = xcd_contiguous(blockIdx.x, gridDim.x);
    const int item = (int)(wg % igroups) * WAVES + wave; wg /= igroups;
    const int mchunk = wg % P.mchunks; wg /= P.mchunks;
    const int g = wg % P.G, split = wg / P.G;
    // the item's channel tile: segments are the intersections of the convolution group with deformable groups
    const int tgroups = (P.kV + TP - 1) / TP, tap0 = item % tgroups * TP, ts = QUAD ? j % 8 / (LW / 4) : j / LW;      // ts: this lane's tap among them
    int z = item / tgroups, dg, c0 = 0, ce = 0;
    bool works = false;
    for (dg = g * P.Cg / P.cpg; dg <= ((g + 1) * P.Cg - 1) / P.cpg; ++dg) {
        const int cb = max(g * P.Cg, dg * P.cpg);
        ce = min((g + 1) * P.Cg, (dg + 1) * P.cpg);
        const int nt = (ce - cb + TC - 1) / TC;
        if (z < nt) { c0 = cb + z * TC; works = true; break; }
        z -= nt;
    }
    if (!works) dg = 0;         // (a wavefront without an item helps with the rows)

    // taps whose geometry this lane works out (lane groups take turns), clamped to legal ones
    int gtap[GT], kd[GT][ND];
#pragma unroll
    for (int u = 0; u < GT; ++u) {
        gtap[u] = min(tap0 + (TP > 1 ? 2 * u + q : 0), P.kV - 1);
        int kk[ND];
        decode_tap<ND>(P, gtap[u], kk);
#pragma unroll
        for (int a = 0; a < ND; ++a) kd[u][a] = kk[a] * P.dil[slot<ND>(a)];
    }

    const int m_base = mchunk * MT * TN;
    constexpr int CL = QUAD ? 4 * CT : CT;                      // channels that a lane loads
    const int cq = QUAD ? j % 8 % (LW / 4) : j % LW;
    const unsigned cj = (unsigned)min(c0 + cq * CL, P.C_in - CL);          // clamped: lanes past the segment still load legally
    auto column = [&](int u) { return QUAD ? cq * CL + u * 4 + j / 8 : cq * CT + u; };      // channel of this lane's column of tile u
    // 32-bit byte offsets from the sample's base (the host checks that a sample of either tensor stays below 4 GiB)
    const unsigned cjB = cj * (unsigned)sizeof(S), cinB = (unsigned)P.C_in * (unsigned)sizeof(S);
    unsigned strB[ND];                                          // from a corner to the next along an axis
    {
        unsigned s = cinB;
#pragma unroll
        for (int a = ND - 1; a >= 0; --a) {
            strB[a] = P.in[slot<ND>(a)] > 1 ? s : 0u;
            s *= (unsigned)P.in[slot<ND>(a)];
        }
    }
    // what this thread copies of a step's rows: 16 bytes each, rows past M as row M - 1
    constexpr int NROW = MT * NP * 64, NA = (NROW + WG - 1) / WG;
    unsigned r_at[NA], r_q[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int x = i * WG + threadIdx.x, m = x % (MT * TN), pq = min(x / (MT * TN), NP * 2 - 1);
        r_at[i] = ((unsigned)(pq / 2) * P.C_out + g * P.M + min(m_base + m, P.M - 1)) * 16u;
        r_q[i] = pq & 1;
    }

    typename MM::Acc acc[CT][MT];
    const int slabs_per_sample = (int)(row_steps(P.outV) / 2), nslabs = P.N * slabs_per_sample;
    // the splits of an XCD take turns in a range of the slabs of their own (against all splits in turn over all slabs: 64 -> 64 channels in
    // 3-D 597 -> 587 us, 128 -> 128 with stride 2 907 -> 838: fewer reads past the L2)
    const int runs = min(P.nsplit, 8), run = (int)((unsigned)split * runs / (unsigned)P.nsplit);
    const int s0 = (run * P.nsplit + runs - 1) / runs, s1 = ((run + 1) * P.nsplit + runs - 1) / runs;      // its splits
    const int first = (int)((long long)nslabs * s0 / P.nsplit) + split - s0, last = (int)((long long)nslabs * s1 / P.nsplit), turn = s1 - s0;
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[u][mt] = acc_zero<T>();
    // A slab's positions are four octets.  In 3-D of float32, which reads a corner's channels dword by dword and waits for the L1: of a run of 4 * S octets
    // -- about four rows of the output -- slab r takes octets r, r + S, r + 2 S, r + 3 S, a block of positions, whose samples share more lines than
    // those of 32 positions in a row; the octets behind the last whole run in order.  (Steps of 64 -> 64, rows of 56: 2436 -> 2406 us, 128 -> 128
    // at stride 1 2 2 4484 -> 4461.  2-D waits less for the L1 and loses the arithmetic: 256 -> 256 861 -> 870, no offsets 90 -> 92.)
    constexpr bool BLOCKS = ND == 3 && sizeof(S) == 4 && !PLAIN;
    const int S4 = BLOCKS ? max((P.out[2].d + 4) / 8, 1) : 1, runs4 = BLOCKS ? slabs_per_sample / S4 * S4 : 0;
    auto first_octet = [&](int slab, int& stride) {     // of a slab of a sample
        stride = BLOCKS && slab < runs4 ? S4 : 1;
        return BLOCKS && slab < runs4 ? slab / S4 * S4 * 4 + slab % S4 : slab * 4;
    };
    const unsigned octet_bytes = (unsigned)(NP * P.C_out * 16);
    const char* const row0 = reinterpret_cast<const char*>(rows);
    Vec rv[NA];
    auto load_rows = [&](int slab, int st) {
        const int n = slab / slabs_per_sample;
        int stride;
        const int oct = first_octet(slab - n * slabs_per_sample, stride);
        const char* ap = row0 + ((size_t)n * slabs_per_sample * 4 + oct + 2 * st * stride) * octet_bytes;
        const unsigned next = (unsigned)stride * octet_bytes;
#pragma unroll
        for (int i = 0; i < NA; ++i) rv[i] = *reinterpret_cast<const Vec*>(ap + (r_at[i] + (r_q[i] ? next : 0u)));
    };
    auto slab_position = [&](int slab, int at) {        // position `at` (0 .. 31) of a slab of all samples, in its sample
        int stride;
        const int oct = first_octet(slab % slabs_per_sample, stride);
        return (unsigned)(oct + at / 8 * stride) * 8u + (unsigned)(at % 8);
    };
    auto put_rows = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
            if ((i + 1) * WG <= NROW || i * WG + threadIdx.x < NROW) *reinterpret_cast<Vec*>(sRow[buf] + (i * WG + threadIdx.x) * 16) = rv[i];
    };
    T offv[GT][ND];
    auto load_off = [&](int slab) {
        const int n = slab / slabs_per_sample;
        const unsigned posc = min(slab_position(slab, j), P.outV - 1);
        const S* off_n = PLAIN ? nullptr : off + ((size_t)n * P.DG + dg) * P.kV * ND * P.outV;
#pragma unroll
        for (int u = 0; u < GT; ++u)
#pragma unroll
            for (int a = 0; a < ND; ++a) offv[u][a] = PLAIN ? 0.f : Store<S>::ld(off_n[((size_t)gtap[u] * ND + a) * P.outV + posc]);
    };
    const T sgn = split & 1 ? -1.f : 1.f;               // of this split's samples
    if (first < last) {
        load_off(first);
        load_rows(first, 0);
        put_rows(0);
    }
    __syncthreads();
    for (int slab = first; slab < last; slab += turn) {
        const int n = slab / slabs_per_sample;
        const char* in_n = reinterpret_cast<const char*>(in_cl + (size_t)n * P.inV * P.C_in);        // scalar bases
        const int next_slab = min(slab + turn, last - 1);
        const unsigned pos = slab_position(slab, j);
        const bool valid = pos < P.outV;
        const unsigned posc = valid ? pos : P.outV - 1;
        int o[ND];
        decode_pos<ND>(P, posc, o);
        // LDS operations of one wavefront execute in order; the fences only pin the compiler
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < GT; ++u) {
            bool live = valid;
            T f[ND];
            unsigned base = 0;
#pragma unroll
            for (int a = 0; a < ND; ++a) {
                const int sa = slot<ND>(a);
                const T p = (T)(o[a] * P.stride[sa] - P.pad[sa] + kd[u][a]) + offv[u][a];
                const T pc = __builtin_amdgcn_fmed3f(p, 0.f, (T)(P.in[sa] - 1));
                live = live && fabsf(p - pc) < 1.f;                 // -1 < p < size, false for NaN
                int lo = (int)pc;
                if constexpr (!PLAIN) lo = min(lo, max(P.in[sa] - 2, 0));
                f[a] = pc - (T)lo;
                base = base * (unsigned)P.in[sa] + (unsigned)lo;
            }
            if (TP > 1 || q == 0) {
                const int row = TP > 1 ? 2 * u + q : 0;
                T cw[NC];                              // multiplied in the reference's order (w_l * w_h * w_w)
                if constexpr (ND == 3) {
                    const T fl = f[0], gl = 1.f - fl, fh = f[1], gh = 1.f - fh, fw = f[2], gw = 1.f - fw;
                    cw[0] = gl * gh * gw; cw[1] = gl * gh * fw; cw[2] = gl * fh * gw; cw[3] = gl * fh * fw;
                    cw[4] = fl * gh * gw; cw[5] = fl * gh * fw; cw[6] = fl * fh * gw; cw[7] = fl * fh * fw;
                } else {
                    const T fh = f[0], gh = 1.f - fh, fw = f[1], gw = 1.f - fw;
                    cw[0] = gh * gw; cw[1] = gh * fw; cw[2] = fh * gw; cw[3] = fh * fw;
                }
                sIdx[wave][row][j] = live ? base * cinB : 0u;
#pragma unroll
                for (int i = 0; i < NR; ++i) sCw[wave][row][j][i] = !live ? 0.f : PLAIN ? sgn : sgn * cw[i];
            }
        }
        load_off(next_slab);                            // travel through this slab
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        const char* corner[NR];                     // scalar
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            size_t d = 0;
#pragma unroll
            for (int a = 0; a < ND; ++a)
                if ((i >> (ND - 1 - a)) & 1) d += strB[a];
            corner[i] = in_n + d;
        }
        // one position (QUAD: four of the lane group's eight, one to every eight lanes) after the other; the next one's record and corner values are
        // on their way while this one is added up
        constexpr int PB = QUAD ? 2 : 8;            // such turns to a step
        constexpr int NB = QUAD && NR > 4 ? 4 : NR, HB = NR / NB;       // corners at a time, for the registers
        typedef typename std::conditional<QUAD, Quad, typename std::conditional<CT == 1, T, unsigned>::type>::type Word;
        Word cn[NB];
        T wn[NB];
        auto fetch = [&](int k) {
            const int h = k % HB, e = k / HB % PB;
            const int pp = k / HB / PB * 16 + q * 8 + (QUAD ? e * 4 + j / 8 : e);          // position of the slab this lane works on
            const unsigned at = sIdx[wave][ts][pp] + cjB;
#pragma unroll
            for (int i = 0; i < NB; ++i) wn[i] = sCw[wave][ts][pp][h * NB + i];
#pragma unroll
            for (int i = 0; i < NB; ++i) cn[i] = *reinterpret_cast<const Word*>(corner[h * NB + i] + at);
        };
        if (works) fetch(0);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            load_rows(st == 0 ? slab : next_slab, st ^ 1);
            if (works) {
                float val[CT][8];
#pragma unroll
                for (int e = 0; e < PB; ++e) {
#pragma unroll
                    for (int h = 0; h < HB; ++h) {
                        const int k = (st * PB + e) * HB + h;
                        Word cc[NB];
                        T wc[NB];
#pragma unroll
                        for (int i = 0; i < NB; ++i) { cc[i] = cn[i]; wc[i] = wn[i]; }
                        if (k + 1 < 2 * PB * HB) fetch(k + 1);
                        __builtin_amdgcn_sched_barrier(0);      // the next loads are issued before this turn's arithmetic
                        // weighted corner sum, as the reference's sampler forms it
#pragma unroll
                        for (int u = 0; u < CL; ++u) {
                            T& v = QUAD ? val[u / 4][e * 4 + u % 4] : val[u][e];
                            v = h ? v + wc[0] * channel_of<S>(cc[0], u) : wc[0] * channel_of<S>(cc[0], u);
#pragma unroll
                            for (int i = 1; i < NB; ++i) v += wc[i] * channel_of<S>(cc[i], u);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if constexpr (QUAD) {
#pragma unroll
                        for (int u = 0; u < CT; ++u) swap_lanes_registers(val[u] + e * 4);
                    }
                }
                // B[k = position][col = channel j]: weight 0 where there is no sample and past the end.  A row of A only reaches
                // its own row of the tile and a column of B its own column, and rows past M / columns past the segment are not stored.
                Vec b8[CT][NP];
#pragma unroll
                for (int u = 0; u < CT; ++u) PT::split(val[u], b8[u]);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    Vec a8[1][NP];
#pragma unroll
                    for (int x = 0; x < NP; ++x) a8[0][x] = *reinterpret_cast<const Vec*>(sRow[st] + ((x * 2 + q) * MT * TN + mt * TN + j) * 16);
#pragma unroll
                    for (int u = 0; u < CT; ++u) {
                        if constexpr (NP > 1) {
                            typename MM::Acc sum[1] = {acc_zero<T>()};
                            mma_parts<S, 1>(a8, b8[u], sum);
                            acc[u][mt] += sum[0];
                        } else
                            mma_parts<S, 1>(a8, b8[u], &acc[u][mt]);
                    }
                }
            }
            put_rows(st ^ 1);
            __syncthreads();
        }
    }
    bool stands = true;
#pragma unroll
    for (int u = 0; u < CT; ++u) stands = stands && results_stand<MT, S>(acc[u]);
    const bool redo = works && __any(!stands);
    // One row tile from the values themselves, two positions at a time, with the reference's corners.  (Its own accumulator, after
    // the loop above: a second loop over `acc` doubled the registers of the kernel.)
    const int tap = tap0 + ts;                          // of this lane's column
    auto exact_tile = [&](int u, int mt) {
        typename MM::Acc x = acc_zero<T>();
        int kk[ND], kx[ND];
        decode_tap<ND>(P, min(tap, P.kV - 1), kk);
#pragma unroll
        for (int a = 0; a < ND; ++a) kx[a] = kk[a] * P.dil[slot<ND>(a)];
        for (int slab = first; slab < last; slab += turn) {
            const int n = slab / slabs_per_sample;
            const S* off_n = PLAIN ? nullptr : off + (((size_t)n * P.DG + dg) * P.kV + min(tap, P.kV - 1)) * ND * P.outV;
            const char* in_n = reinterpret_cast<const char*>(in_cl + (size_t)n * P.inV * P.C_in);
#pragma unroll 1
            for (int ks = 0; ks < TN; ks += 2) {
                const unsigned pos = slab_position(slab, ks + q), posc = min(pos, P.outV - 1);
                int o[ND], ib[ND];
                decode_pos<ND>(P, posc, o);
#pragma unroll
                for (int a = 0; a < ND; ++a) ib[a] = o[a] * P.stride[slot<ND>(a)] - P.pad[slot<ND>(a)];
                T ofx[ND];
#pragma unroll
                for (int a = 0; a < ND; ++a) ofx[a] = PLAIN ? 0.f : Store<S>::ld(off_n[(size_t)a * P.outV + posc]);
                TapGeo<T, ND> t;
                tap_setup_noidx<T, ND>(P, ofx, ib, kx, t);
                const bool live = pos < P.outV && t.inside;
                unsigned cb[NC];
                tap_corner_offsets<T, ND>(P, t, live, cinB, cb);
                T v = 0.f;
#pragma unroll
                for (int i = 0; i < NR; ++i) {
                    T w = 1.f;
#pragma unroll
                    for (int a = 0; a < ND; ++a) w *= PLAIN ? 1.f : (i >> (ND - 1 - a)) & 1 ? t.f[a] : 1.f - t.f[a];
                    v += w * Store<S>::ld(*reinterpret_cast<const S*>(in_n + (cb[i] + (unsigned)min(c0 + column(u), P.C_in - 1) * (unsigned)sizeof(S))));
                }
                if constexpr (CT > 1) v = (T)(typename PT::Elem)v;         // rounded like the operand
                const T b = live ? v : 0.f;
                const int m = min(m_base + mt * TN + j, P.M - 1);
                const T av = pos < P.outV ? Store<S>::ld(gout[((size_t)n * P.C_out + g * P.M + m) * P.outV + posc]) : 0.f;
                x = MM::mma(av, b, x);
            }
        }
        return x;
    };

    if (!works) return;                                 // (uniform for the wavefront)
    T* pt = partial + ((size_t)split * P.kV + tap) * P.C_out * P.Cg + (size_t)g * P.M * P.Cg + (c0 - g * P.Cg);
#pragma unroll
    for (int u = 0; u < CT; ++u)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        typename MM::Acc x = acc[u][mt] * sgn;
        if (__builtin_expect(redo, 0)) x = exact_tile(u, mt);
#pragma unroll
        for (int r = 0; r < MM::NACC; ++r) {
            const int m = m_base + mt * TN + MM::row(r, q);
            if (m < P.M && c0 + column(u) < ce && tap < P.kV) pt[(size_t)m * P.Cg + column(u)] = x[r];
        }
    }
}

// 16-byte loads (QUAD) where every lane's channels of a voxel are aligned to them, but not for
// - float32 in 3-D (see the top of the file),
// - bfloat16 in 3-D with eight lanes to a tap and more than one row tile, which spills 69 registers with them: backward passes to the weight of 16 such layers, us with 4 bytes
//   to a lane : 16 -- 64 -> 64 in groups of 8, 4 x 16 x 28 x 28, 268 : 384; 16 -> 48 in groups of 8, 4 x 16 x 56 x 56, 210 : 351; never less than 1.19 times as long.  (One
//   row tile 1.02 to 1.25 times as fast with 16, binary16 1.00 to 1.22.)
// float32 in 2-D with fewer than 32 lanes to a tap, 680 layers: 0.95 to 1.28 times as fast with them, 1.01 on average, one row tile 1.08; no line by channels or
// row tiles does better.  16-bit storage in 2-D with fewer than 32 lanes: 1.00 to 1.30, 1.05 on average.
template <int ND, typename S>
inline bool split_quad(const Params& P, int MT, int LW) {
    constexpr int CL = 16 / sizeof(S);
    if (P.C_in % CL || P.cpg % CL || P.Cg % CL || (ND == 3 && sizeof(S) == 4)) return false;
    return !(ND == 3 && std::is_same<S, Bf16>::value && LW == 8 && MT > 1);
}

// Estimated time of a split, in us: a wavefront's share of the slabs, 4 to a slab, times the rounds of workgroups -- of less than one, the
// part a workgroup takes when its CU holds no other, and the rest with what shares the CU -- and the partial tiles (of `one` bytes a split).  Backward passes
// of 60 layers, the other line's time over this one's: 0.2 for 0.4 1.03 (at worst 1.13), 0.6 1.013 (1.07), 1 1.005 (1.04); 1 for 4 1.019 (1.12), 2 1.005,
// 8 and 16 1.001 (1.03).  A plain convolution is planned by the occupancy of the kernel with offsets (24 layers by its own: 1.0015, at worst 1.02).
struct SplitCost { double slabs, tiles; int nsplit; };  // nsplit 0: no room
inline SplitCost split_cost(double workgroups, double resident, long long nslabs, long long most, size_t one) {
    SplitCost best = {0, 0, 0};
    if (most > 256) most = 256;
    if (most > nslabs) most = nslabs;
    for (long long s = 1; s <= most; ++s) {
        const double load = workgroups * (double)s / resident, rounds = load > 1 ? ceil(load) : 0.4 + 0.6 * load;
        const SplitCost c = {(double)((nslabs + s - 1) / s) * rounds * 4, (double)s * (double)one * 2 / 8e6, (int)s};
        if (s == 1 || c.slabs + c.tiles < best.slabs + best.tiles) best = c;
    }
    return best;
}
// Whether eight row tiles to a workgroup are faster than four, by the estimates of either: a slab of eight, two wavefronts to a SIMD, takes 1.18 times as long as one of four, three to a
// SIMD, in 3-D and 1.22 times in 2-D, where the corner reads are a smaller part.  Backward passes to the weight of 504 layers of more than 128 output channels: by this line 1.0022
// times the time of the better one on average, always eight 1.013 (at worst 1.22: 950 -> 415 to each of two groups, 3x3, two samples of 26 x 20, 233 us : 284; 86 -> 249, 3x3, two of 67 x 99,
// 77 : 91; 128 -> 256, 1x1x1, 4 x 16 x 56 x 56, 384 : 406), always four 1.08 (64 -> 256, 3x3x3, 4 x 16 x 56 x 56, 1727 : 1415).
inline bool eight_tiles_pay(int nd, const SplitCost& four, const SplitCost& eight) {
    return eight.nsplit > 0 && eight.slabs * (nd == 3 ? 1.18 : 1.22) + eight.tiles < four.slabs + four.tiles;
}

}  // namespace dcn
