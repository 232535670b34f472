// Forward kernel of the float32 and 16-bit operators: input halo in LDS, contraction on the 16-bit
// matrix instructions.
//
//   out[n][g*M + m][pos] = sum_{cl,tap} W[g*M+m][cl][tap] * sample(in[n][g*Cg+cl], tap, pos)  (+ bias)
//
// replaces deformable_im2col + the per-group Sgemm of the reference
// (deform3d/lib/deform_conv3d_cuda.cpp:110-148, deform2d_double/lib/deform_conv2d_cuda.cpp:102-138).
//
// Contraction of float32 operands.  A float32 value is the exact sum of three bfloat16 values: the
// value rounded to bfloat16, the remainder rounded to bfloat16, and what is left (24 significant bits
// = 3 x 8; each remainder is formed without rounding; values from 2^-110 on, see below).  A product of two
// values is then nine products of parts, each exact in float32, of which the three smallest (below 2^-24 of the
// product together) are left out; the other six are summed by v_mfma_f32_32x32x16_bf16 into float32 accumulators,
// smallest first.  Against float64, sums of 64 / 576 / 6912 products of N(0, 1) values are off by 6.5e-8 / 1.0e-7 /
// 3.4e-7 (2-norm), by v_mfma_f32_32x32x2_f32, which rounds after every second product where this rounds
// after every sixteenth, by 9.2e-8 / 2.4e-7 / 5.2e-7.  Six instructions reduce over 16 slots in 81 ns per SIMD
// (13.5 each) where eight float32 ones take 216 to 239 ns, and unlike those they run next to vector instructions.
// Operands without such parts: a workgroup works its block out once more through the float32
// instructions, on the weights as they are, when a result
//   - is not finite (inf - inf in the parts; this also gives an overflow of the parts the float32 meaning), or
//   - lies below 2^-80 without being zero.  The third part of a value below 2^-110 is subnormal and loses bits,
//     up to 2^-134 per value: more than float32 sums round away only where a result is below 2^-110 times
//     the sum of the other operand's magnitudes.  With sums of up to 2^30 that never goes unnoticed (x around
//     2^-116, weights around 2^10: 3.6e-6 from float64 without the second look, 4e-7 with it).
//     Samples below 2^-133 (float32 subnormals) count as zero where the result is not looked at again.
//
// Lane roles.  A wavefront owns 32 output positions; lane (j, q) works on position j and supplies
// eight of the 16 reduction slots of an instruction: eight channels of tap tg*2 + q.  Every lane derives
// the geometry of ONE (tap, position) per tap pair and no two lanes repeat each other's work; the halo
// holds four channels of a voxel in 16 consecutive bytes, so that one wide LDS read per corner fetches
// four of the lane's values.
#pragma once
#include <limits>
#include "dcn_kernels.h"
#include "dcn_forward.h"

namespace dcn {

constexpr int FG = 8;              // channels per reduction group: what a lane supplies to one matrix instruction

// The 16-bit matrix instruction with 16 reduction slots, and how a lane's eight values become operands.
template <typename S> struct Parts;
template <> struct Parts<float> {
    static constexpr int NP = 3;   // bfloat16 parts of a value
    typedef __bf16 Vec __attribute__((ext_vector_type(8)));
    static __device__ inline void split(const float v[8], Vec p[NP]) {
        typedef __bf16 B2 __attribute__((ext_vector_type(2)));
        typedef float F2 __attribute__((ext_vector_type(2)));
        typedef unsigned U4 __attribute__((ext_vector_type(4)));
        U4 out[NP];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
            for (int k = 0; k < NP; ++k) {
                const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(F2{a, b}, B2));
                out[k][i] = u;
                a -= __uint_as_float(u << 16);
                b -= __uint_as_float(u & 0xffff0000u);
            }
        }
#pragma unroll
        for (int k = 0; k < NP; ++k) p[k] = __builtin_bit_cast(Vec, out[k]);
    }
    // parts of one value for the packed weights; infinities and NaN stay in the first part, and so that
    // a value near the largest float does not round to infinity its first part is then cut off instead
    // nor does a nonzero weight round to zero: results made of it are too small not to be looked at again
    static __device__ inline void split1(float v, __bf16 p[NP]) {
        p[0] = (__bf16)v;
        if (v != 0.f && (float)p[0] == 0.f) p[0] = (__bf16)copysignf(0x1p-133f, v);
        if (!(fabsf((float)p[0]) <= std::numeric_limits<float>::max())) {
            if (!(fabsf(v) <= std::numeric_limits<float>::max())) { p[1] = p[2] = (__bf16)0.f; return; }
            p[0] = (__bf16)__uint_as_float(__float_as_uint(v) & 0xffff0000u);
        }
        p[1] = (__bf16)(v - (float)p[0]);
        p[2] = (__bf16)((v - (float)p[0]) - (float)p[1]);
    }
    typedef __bf16 Elem;
    static __device__ inline Mma<float>::Acc mma(Vec a, Vec b, Mma<float>::Acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Parts<Bf16> {
    static constexpr int NP = 1;
    typedef __bf16 Vec __attribute__((ext_vector_type(8)));
    typedef __bf16 Elem;
    static __device__ inline void split(const float v[8], Vec p[NP]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) p[0][e] = (__bf16)v[e];            // round to nearest even
    }
    static __device__ inline void split1(Bf16 v, __bf16 p[NP]) { p[0] = __builtin_bit_cast(__bf16, v.bits); }
    static __device__ inline Mma<float>::Acc mma(Vec a, Vec b, Mma<float>::Acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Parts<Fp16> {
    static constexpr int NP = 1;
    typedef _Float16 Vec __attribute__((ext_vector_type(8)));
    typedef _Float16 Elem;
    static __device__ inline void split(const float v[8], Vec p[NP]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) p[0][e] = (_Float16)v[e];
    }
    static __device__ inline void split1(Fp16 v, _Float16 p[NP]) { p[0] = v.v; }
    static __device__ inline Mma<float>::Acc mma(Vec a, Vec b, Mma<float>::Acc c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
// acc[mt] += A[mt] * B for MT row tiles: the products of parts i, j with i + j < NP, smallest first
template <typename S, int MT>
__device__ inline void mma_parts(const typename Parts<S>::Vec a[MT][Parts<S>::NP], const typename Parts<S>::Vec b[Parts<S>::NP],
                                 Mma<float>::Acc acc[MT]) {
    constexpr int NP = Parts<S>::NP;
#pragma unroll
    for (int sum = NP - 1; sum >= 0; --sum)
#pragma unroll
        for (int i = 0; i <= sum; ++i)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] = Parts<S>::mma(a[mt][i], b[sum - i], acc[mt]);
}

// Packed weights: one slab per group of eight channels (groups start at the first channel of a
// segment and at every eighth after it), in the order the lanes consume them:
//   Wq[slab][tap pair][row tile][part][q][j][e] = part of W[m = tile*32 + j][channel = first + e][tap = tg*2 + q]
// zero past M, past the last tap and past the segment.  An operand is 16 contiguous bytes of a lane and
// 1 KB of a wavefront.
template <typename S>
__host__ __device__ inline size_t split_slab_elems(int kV, int Mp) {
    return (size_t)((kV + 1) / 2) * Mp * 2 * FG * Parts<S>::NP;
}

// weight of output channel m and input channel cl of group g
template <typename S> __device__ inline S weight_at(const Params& P, const S* __restrict__ W, int g, int m, size_t cl, int tap) {
    return P.transposed ? W[(((size_t)g * P.Cg + cl) * P.M + m) * P.kV + (P.kV - 1 - tap)] : W[(((size_t)g * P.M + m) * P.Cg + cl) * P.kV + tap];
}

// A wavefront per operand.  With pc.sel set the launch has one block more, which chooses the
// halo plan from the offsets.
template <typename S>
__global__ __launch_bounds__(256) void pack_split_weight_kernel(Params P, const S* __restrict__ W, typename Parts<S>::Elem* __restrict__ Wq,
                                                                PlanChoice pc, const S* __restrict__ off, size_t n_off) {
    touch_arguments<sizeof(Params) + sizeof(PlanChoice) + 24>();
    using PT = Parts<S>;
    constexpr int TN = 32, NP = PT::NP;
    const unsigned pack_blocks = pc.sel ? gridDim.x - 1 : gridDim.x;
    if (blockIdx.x == pack_blocks) {
        choose_plan(pc, off, n_off);
        return;
    }
    const unsigned mtiles = P.Mp / TN, ntg = (P.kV + 1) / 2, per_slab = ntg * mtiles;       // wavefronts of a slab
    const unsigned total = (unsigned)chunk_candidates<FG>(P.cpg, P.Cg, P.C_in) * per_slab;
    const unsigned lane = threadIdx.x & 63;
    for (unsigned w = (unsigned)__builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); w < total; w += pack_blocks * 4) {      // uniform for a wavefront
        const unsigned cand = w / per_slab, r = w - cand * per_slab;
        const int c0 = chunk_candidate<FG>(P.cpg, P.Cg, (int)cand);                 // candidate first channel of a group
        const int g = c0 / P.Cg, dg = c0 / P.cpg, seg_b = max(dg * P.cpg, g * P.Cg), seg_e = min((dg + 1) * P.cpg, (g + 1) * P.Cg);
        if ((c0 - seg_b) % FG) continue;
        const int tg = (int)(r / mtiles), tile = (int)r - tg * (int)mtiles;
        const int m = tile * TN + lane % TN, tap = tg * 2 + lane / TN;
        // (no load is masked: a masked one is waited for on its own)
        S v[FG];
#pragma unroll
        for (int e = 0; e < FG; ++e) v[e] = weight_at<S>(P, W, g, min(m, P.M - 1), (size_t)(min(c0 + e, seg_e - 1) - g * P.Cg), min(tap, P.kV - 1));
        typename PT::Vec part[NP];
#pragma unroll
        for (int e = 0; e < FG; ++e) {
            typename PT::Elem p[NP];
            PT::split1(m < P.M && tap < P.kV && c0 + e < seg_e ? v[e] : S(), p);
#pragma unroll
            for (int k = 0; k < NP; ++k) part[k][e] = p[k];
        }
        typename PT::Vec* dst = reinterpret_cast<typename PT::Vec*>(Wq) + ((size_t)chunk_slot<FG>(P.cpg, P.Cg, c0) * per_slab + r) * NP * 64 + lane;
#pragma unroll
        for (int k = 0; k < NP; ++k) dst[k * 64] = part[k];
    }
}

// Offset of halo voxel v inside a channel of the input, ~0u outside the volume.  The two divisions
// are float multiplications by a reciprocal: half a voxel of slack is far more than their rounding for the few
// thousand voxels of a halo.
template <int ND>
__device__ inline unsigned halo_voxel(const Params& P, const HaloPlan& H, const TileGeo<ND>& tg, int v, float inv1, float inv2) {
    const int r = (int)(((float)v + 0.5f) * inv2);
    int c[ND];
    c[ND - 1] = v - __mul24(r, H.hext[2]);
    if constexpr (ND == 3) {
        c[0] = (int)(((float)r + 0.5f) * inv1);
        c[1] = r - __mul24(c[0], H.hext[1]);
    } else
        c[0] = r;
    bool inb = true;
    unsigned lin = 0;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        c[a] += tg.hb[a];
        inb = inb && (unsigned)c[a] < (unsigned)P.in[slot<ND>(a)];
        lin = lin * (unsigned)P.in[slot<ND>(a)] + (unsigned)c[a];
    }
    return inb ? lin : ~0u;
}

// What a workgroup of a forward launch works on: units are (block of positions, group, output-channel
// chunk), workgroups of one tile are neighbours in an XCD-contiguous order.  The launch splits units as
// described at forward_quad_kernel: csplit > 1 and whole = 0, every unit; whole > 0, the units from
// `whole` on, in the two runs of TailSplit.
struct ForwardUnit {
    unsigned wg;                // unit
    unsigned pslot;             // which partial sum of the split runs
    int cz;                     // this workgroup takes every cs-th channel pass, from the cz-th on
    Div cs;
    int cch;                    // channels per LDS pass
    bool split;
};
__device__ inline ForwardUnit forward_unit(int cchunk, const Div& csplit, unsigned whole, const TailSplit& ts) {
    ForwardUnit u;
    u.pslot = 0;
    u.cz = 0;
    u.cs = csplit;
    u.cch = cchunk;
    u.split = csplit.d > 1 && blockIdx.x >= whole;
    if (!u.split) {
        u.wg = xcd_contiguous(blockIdx.x, csplit.d > 1 ? whole : gridDim.x);
        u.cs = Div{};                                      // (not divided by: one workgroup takes every pass)
        u.cs.d = 1;
        return u;
    }
    const unsigned rel = blockIdx.x - whole, all = gridDim.x - whole;
    const unsigned wgsA = ts.splitB.d ? ts.unitsA * (unsigned)csplit.d : all;
    unsigned first = whole, r;
    if (rel < wgsA) {
        r = xcd_contiguous(rel, wgsA);
        u.pslot = r;
    } else {
        r = xcd_contiguous(rel - wgsA, all - wgsA);
        u.cs = ts.splitB;
        first = whole + ts.unitsA;
        u.pslot = wgsA + r;
        u.cch = min(cchunk, ts.cchB);
    }
    const unsigned unit = r / u.cs;
    u.wg = first + unit;
    u.cz = (int)(r - unit * (unsigned)u.cs.d);
    return u;
}

// The halo in LDS: 16-byte cells [cell plane][halo voxel] that hold the next few channels of a voxel in
// their storage format, four float32 or eight 16-bit ones: one wide read fetches them all.  (16-bit values
// are widened after the read: half the LDS reads and twice the channels per pass of a float halo.)
template <typename S> struct HaloCell {
    static constexpr int CH = 16 / sizeof(S);
    typedef typename std::conditional<sizeof(S) == 4, float, typename Parts<S>::Elem>::type V;
    typedef V Vec __attribute__((ext_vector_type(CH)));
    static __device__ inline V raw(S v) { return __builtin_bit_cast(V, v); }
};

// Stages `nch` channels of the halo, planes of hstride cells; missing channels of a short last group
// and voxels outside the volume hold zero.  Returns whether the thread met a non-finite value (CHECK).
template <int ND, int WGS, bool CHECK, typename S>
__device__ inline bool stage_halo(const Params& P, const HaloPlan& H, const TileGeo<ND>& tg, const S* __restrict__ chan0, int nch,
                                  typename HaloCell<S>::Vec* __restrict__ sIn) {
    constexpr int CH = HaloCell<S>::CH;
    // an item is a cell: consecutive threads take consecutive voxels
    const int items = (nch + CH - 1) / CH * H.hvol;
    const float inv2 = __builtin_amdgcn_rcpf((float)H.hext[2]), inv1 = __builtin_amdgcn_rcpf((float)H.hext[1]), inv = __builtin_amdgcn_rcpf((float)H.hvol);
    const size_t step = (size_t)P.inV * sizeof(S);
    // Items of a thread in flight, the last ones too: a pass waits for memory ceil(items / U) times.  (Four in a loop unrolled so, and the remainder one by
    // one: 256 -> 256, 2-D, steps 880 -> 858 us, the ragged 48 -> 80 in 3-D 398 -> 390.  Of 128 -> 128 at stride 1 2 2, eight wavefronts, 17 items: 2, 3, 4, 6
    // in flight 4535, 4497, 4511, 4476; 64 -> 64 in 3-D, sixteen wavefronts, inference: 469, 471, 481, 471.  With six, layers of few channels repeat more loads
    // than they have: inference of 10 -> 41 in groups of 5, 3x3, 4 x 174 x 138, 53.4 us before any of this, 58.8 with six, 53.3 with three; 44 -> 43 in groups of 11,
    // 1x1x1, 8 x 30 x 28 x 53, 166, 182, 167; 70 drawn layers 1.046 times as fast as before with six, 1.058 with three.)
    constexpr int U = 3;
    bool bad = false;
    // (no load is masked: a masked one is waited for on its own; past the last item and past the last channel a load is repeated)
    auto stage = [&](int it0, auto count) {
        constexpr int C = decltype(count)::value;
        typename HaloCell<S>::Vec cell[C];
        int grp[C], v[C];
        bool there[C];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const int it = min(it0 + u * WGS, items - 1);
            grp[u] = (int)(((float)it + 0.5f) * inv);
            v[u] = it - __mul24(grp[u], H.hvol);
            const unsigned t = halo_voxel<ND>(P, H, tg, v[u], inv1, inv2);
            there[u] = t != ~0u;
            const char* cp = reinterpret_cast<const char*>(chan0) + (size_t)(there[u] ? t : 0u) * sizeof(S) + (size_t)(grp[u] * CH) * step;
            const int last = nch - 1 - grp[u] * CH;             // >= CH - 1 but in a short last group
#pragma unroll
            for (int e = 0; e < CH; ++e) cell[u][e] = HaloCell<S>::raw(*reinterpret_cast<const S*>(cp + (size_t)min(e, last) * step));
        }
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const int last = nch - 1 - grp[u] * CH;
            if constexpr (CHECK) {
#pragma unroll
                for (int e = 0; e < CH; ++e) bad = bad || !(fabsf((float)cell[u][e]) <= std::numeric_limits<float>::max());
            }
#pragma unroll
            for (int e = 0; e < CH; ++e) cell[u][e] = (e <= last && there[u]) ? cell[u][e] : (typename HaloCell<S>::V)0.f;
            if (it0 + u * WGS < items) sIn[(size_t)grp[u] * H.hstride + v[u]] = cell[u];
        }
    };
    for (int it = threadIdx.x; it < items; it += U * WGS) stage(it, std::integral_constant<int, U>{});
    return bad;
}

// Geometry of a lane's (tap, position), following the reference sampler
// (deform3d/lib/deform_conv3d_cuda_kernel.cu:21-26,40-45,123-124) in a branch-free form: the coordinate
// is clamped into [0, size - 1]; low corner = floor, fraction toward the high corner = clamped
// coordinate - floor.  Where the reference collapses the high corner onto the low one (p <= 0,
// p >= size - 1) the fraction is 0, so the corner one step further carries weight 0 and every sample
// uses the same eight (four) cells at fixed strides.
template <int ND> struct SplitTap {
    float pq[ND];               // coordinate
    float cw[1 << ND];          // corner weights w_l * w_h * w_w, all zero without a sample in the halo
    unsigned base;              // low corner's halo cell, 0 without a sample in the halo
    bool near, far;             // sampled from the halo / reaches past it
};
// k0, k1: kernel coordinates of the taps of lane groups 0 and 1 (uniform); rim_far: samples in the
// collapse zones are not taken from the halo.
template <int ND>
__device__ inline void split_geometry(const Params& P, const HaloPlan& H, const TileGeo<ND>& tg, const int ib[ND], int q, const int* k0,
                                      const int* k1, const float* ofs, bool tap_ok, bool rim_far, SplitTap<ND>& t) {
    bool inside = tap_ok, inhalo = true;
    float f[ND];
    int u[ND];
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        const int sa = slot<ND>(a);
        const float top = (float)(P.in[sa] - 1);
        const int kd = k0[a] * P.dil[sa];
        int dk = k1[a] * P.dil[sa] - kd;
        asm volatile("" : "+s"(dk));                            // (scalar arithmetic)
        const float pa = (float)(__mul24(q, dk) + ib[a] + kd) + ofs[a];
        const float pc = __builtin_amdgcn_fmed3f(pa, 0.f, top);
        const float fl = floorf(pc);
        t.pq[a] = pa;
        f[a] = pc - fl;
        inside = inside && fabsf(pa - pc) < 1.f;                // -1 < p < size, false for NaN
        u[a] = (int)fl - tg.hb[a];
        inhalo = inhalo && (unsigned)u[a] < (unsigned)(H.hext[sa] - 1);
    }
    if (rim_far) {
#pragma unroll
        for (int a = 0; a < ND; ++a) inhalo = inhalo && t.pq[a] > 0.f && t.pq[a] < (float)(P.in[slot<ND>(a)] - 1);
    }
    t.near = inside && inhalo;
    t.far = inside && !inhalo;
    unsigned base;
    if constexpr (ND == 3) base = (unsigned)(__mul24(__mul24(u[0], H.hext[1]) + u[1], H.hext[2]) + u[2]);
    else base = (unsigned)(__mul24(u[0], H.hext[2]) + u[1]);
    t.base = t.near ? base : 0u;
    float* cw = t.cw;
    if constexpr (ND == 3) {
        const float fl = t.near ? f[0] : 0.f, gl = t.near ? 1.f - f[0] : 0.f;
        const float fh = f[1], gh = 1.f - fh, fw = f[2], gw = 1.f - fw;
        const float a00 = gl * gh, a01 = gl * fh, a10 = fl * gh, a11 = fl * fh;
        cw[0] = a00 * gw; cw[1] = a00 * fw; cw[2] = a01 * gw; cw[3] = a01 * fw;
        cw[4] = a10 * gw; cw[5] = a10 * fw; cw[6] = a11 * gw; cw[7] = a11 * fw;
    } else {
        const float fh = t.near ? f[0] : 0.f, gh = t.near ? 1.f - f[0] : 0.f, fw = f[1], gw = 1.f - fw;
        cw[0] = gh * gw; cw[1] = gh * fw; cw[2] = fh * gw; cw[3] = fh * fw;
    }
}

// Weighted corner sums of the channels of a cell (element by element: a vector times scalar product
// would hold four copies of every weight).  The sums are formed here, not where the contraction uses
// them, so that one cell's corners are in flight at a time.  row, plane: cells between neighbours along h and l.
// `more` (uniform): also the channels from the fifth on of a 16-bit cell.
template <int ND, typename S>
__device__ inline void cell_sum(const typename HaloCell<S>::Vec* cell, unsigned row, unsigned plane, const float* cw, float* v, bool more) {
    constexpr int NC = 1 << ND, CH = HaloCell<S>::CH;
    typename HaloCell<S>::Vec c[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) c[i] = cell[(i >> 2) * plane + ((i >> 1) & 1) * row + (i & 1)];
#pragma unroll
    for (int h = 0; h < CH; h += 4)
        if (h == 0 || more) {
#pragma unroll
            for (int e = h; e < h + 4; ++e) {
#pragma unroll
                for (int i = 0; i < NC; ++i) v[e] = i ? v[e] + (float)c[i][e] * cw[i] : (float)c[i][e] * cw[i];
            }
#pragma unroll
            for (int e = h; e < h + 4; ++e) asm volatile("" : "+v"(v[e]));
        }
    __builtin_amdgcn_sched_barrier(0);
}
// ... of the eight channels of group grp of a chunk of nch channels
template <int ND, typename S>
__device__ inline void group_sum8(const typename HaloCell<S>::Vec* sIn, unsigned base, int grp, int nch, int hstride, unsigned row,
                                  unsigned plane, const float* cw, float val[FG]) {
    constexpr int CH = HaloCell<S>::CH;
#pragma unroll
    for (int e = 0; e < FG; ++e) val[e] = 0.f;
    const typename HaloCell<S>::Vec* hp = sIn + base + (size_t)grp * (FG / CH) * hstride;
    cell_sum<ND, S>(hp, row, plane, cw, val, grp * FG + 4 < nch);
    if constexpr (CH == 4)
        if (grp * FG + 4 < nch) cell_sum<ND, S>(hp + hstride, row, plane, cw, val + 4, false);
}

// Samples that reach past the halo: val[e] of such lanes = channels c .. c + 7 of the chunk (below nch)
// from global memory, with the reference's corner rule on the same coordinate.
template <int ND, typename S>
__device__ inline void far_values(const Params& P, const SplitTap<ND>& t, const S* __restrict__ chan0, int c, int nch, float val[FG]) {
    constexpr int NC = 1 << ND;
    TapGeo<float, ND> g;
    g.inside = t.far;
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        float pa = t.pq[a];
        asm volatile("" : "+v"(pa));       // (worked out here, not hoisted into the common path)
        const int l = t.far ? (int)pa : 0;
        g.p[a] = pa;
        g.lo[a] = l;
        g.hi[a] = (pa >= (float)(P.in[slot<ND>(a)] - 1) || pa <= 0.f) ? l : l + 1;
        g.f[a] = pa - (float)l;
    }
    tap_corner_idx<float, ND>(P, g);
    // 16 gathers in flight (channel by channel, a layer with one offset in ten beyond its halo waited
    // eight times per step; 32 in 3-D cost the common path its registers)
    constexpr int B = 16 / NC;
#pragma unroll 1
    for (int e0 = 0; e0 < FG; e0 += B) {
        float cc[B][NC];
#pragma unroll
        for (int e = 0; e < B; ++e) {
            const S* ch = chan0 + (size_t)min(c + e0 + e, nch - 1) * P.inV;
#pragma unroll
            for (int i = 0; i < NC; ++i) cc[e][i] = Store<S>::ld(ch[g.idx[i]]);
        }
#pragma unroll
        for (int e = 0; e < B; ++e) {
            const float v = c + e0 + e < nch ? interp<float, ND>(cc[e], g.f) : 0.f;
#pragma unroll
            for (int x = e; x < FG; x += B) val[x] = t.far && x == e0 + e ? v : val[x];
        }
    }
}

// kernel coordinates of the next tap (uniform)
template <int ND>
__device__ inline void next_tap(const Params& P, int k[ND]) {
    int carry = 1;
#pragma unroll
    for (int a = ND - 1; a > 0; --a) {
        k[a] += carry;
        carry = k[a] >= P.k[slot<ND>(a)] ? 1 : 0;
        k[a] = carry ? 0 : k[a];
    }
    k[0] += carry;
}

// offsets of this lane's tap of pair tgi (tap tgi * 2 + q, clamped to a legal tap) at position pos
template <int ND, typename S>
__device__ inline void load_pair_offsets(const Params& P, const S* __restrict__ off_dg, int tgi, int q, unsigned pos, float ofs[ND], bool none) {
    if (none) {                                // (uniform: a plain convolution)
#pragma unroll
        for (int a = 0; a < ND; ++a) ofs[a] = 0.f;
        return;
    }
    const char* ob = reinterpret_cast<const char*>(off_dg + (size_t)tgi * 2 * ND * P.outV);      // uniform
    unsigned lo = ((q && tgi * 2 + 1 < P.kV ? ND * P.outV : 0u) + pos) * (unsigned)sizeof(S);
    asm volatile("" : "+v"(lo));               // (not hoisted into registers that stay live)
#pragma unroll
    for (int a = 0; a < ND; ++a) {
        ofs[a] = Store<S>::ld(*reinterpret_cast<const S*>(ob + lo));
        ob += (size_t)P.outV * sizeof(S);
    }
}

// The contraction of a lane's values on the float32 instructions, one channel of the tap pair at a
// time (results that need a second look).  The weights: in float32 the tensor's own, whose parts may not add
// up to them -- the lane's rows are m0, m0 + 32, ..., its tap is `tap`, its channels cl .. cl + nvalid - 1 of group
// g --, in 16-bit storage the packed ones in `a`.
template <typename S, int MT>
__device__ inline void mma_exact(const Params& P, const S* __restrict__ W, int g, int m0, int tap, size_t cl, const typename Parts<S>::Vec a[MT][Parts<S>::NP],
                                 const float val[FG], bool live, int nvalid, Mma<float>::Acc acc[MT]) {
#pragma unroll 1
    for (int e = 0; e < FG; ++e) {
        float b = 0.f;
#pragma unroll
        for (int x = 0; x < FG; ++x) b = x == e && e < nvalid && live ? val[x] : b;
        if constexpr (sizeof(S) == 2) b = Store<S>::ld(Store<S>::st(b));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float w = 0.f;
            if constexpr (sizeof(S) == 4) {
                const int m = m0 + mt * Mma<float>::TN;
                if (e < nvalid && tap < P.kV && m < P.M) w = weight_at<S>(P, W, g, m, cl + e, tap);
            } else {
#pragma unroll
                for (int x = 0; x < FG; ++x) w = x == e && e < nvalid ? (float)a[mt][0][x] : w;
            }
            acc[mt] = Mma<float>::mma(w, b, acc[mt]);
        }
    }
}

// Whether the lane's results are what they should be: finite (also false when their sum overflows: the workgroup
// then repeats in vain) and, in float32, zero or not too small (see the top of the file).
template <int NT, typename S>
__device__ inline bool results_stand(const Mma<float>::Acc* acc) {
    float s = 0.f;
    unsigned least = ~0u;                               // twice the bits of the least magnitude that is not zero, less one
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < Mma<float>::NACC; ++r) {
            s += fabsf(acc[t][r]);
            if constexpr (sizeof(S) == 4) least = min(least, (__float_as_uint(acc[t][r]) << 1) - 1u);       // (shift-add and half a min3 a value)
        }
    return s <= std::numeric_limits<float>::max() && least >= (__float_as_uint(0x1p-80f) << 1) - 1u;
}

// Writes a 32 x 32 result tile: row m0 + r of group g's output channels (m0 uniform), this lane's position.
// dst: the sample's output, or its partial sums (no bias).
template <typename O, typename S>
__device__ inline void store_tile(const Params& P, O* __restrict__ dst, const S* __restrict__ bias, int g, int m0, int q, unsigned pos,
                                  const Mma<float>::Acc& acc) {
    O* base = dst + ((size_t)g * P.M + m0) * P.outV;                   // uniform
    const unsigned at = (unsigned)q * 4 * P.outV + pos;
    const int rows = P.M - m0 - q * 4;
#pragma unroll
    for (int r = 0; r < Mma<float>::NACC; ++r) {
        const int row = Mma<float>::row(r, 0);
        if (row < rows) {
            float v = acc[r];
            if (bias) v += Store<S>::ld(bias[g * P.M + m0 + row + q * 4]);
            (base + (size_t)row * P.outV)[at] = Store<O>::st(v);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Up to four row tiles (128 output channels) per wavefront, each wavefront sampling its own 32
// positions straight into its operands.  NW wavefronts; dynamic LDS = cchunk * hstride * sizeof(S) bytes,
// cchunk a multiple of eight (or four, float32: half of the reduction slots then stay empty).
// Binding in 3-D: vector instructions, 20 to a matrix instruction, and the LDS reads of the corners beside them (64
// channels, 27 taps, 200 704 positions, 0.49 ms: while a CU holds a workgroup its vector ALUs are busy 74 % of the cycles, its LDS
// 53 %, 63 % of that bank conflicts of random offsets, its matrix units 28 %; 0.64 ms on the float32 instructions).  In
// 2-D: operand latency.
// TS > 1 (layers too small to fill the device otherwise; up to 16): TS wavefronts share 32 positions, each takes a
// contiguous share of a pass's (tap pair, channel group) steps, and their sums meet in LDS -- a step of a lone
// wavefront takes 0.8 to 1.8 us in 2-D, 2.0 to 2.4 us in 3-D (one to four row tiles), most of it latencies, so a small
// layer's time is the length of that chain.
// (up to two row tiles: four wavefronts per SIMD, i.e. at most 128 registers)
template <int ND, int MT, int NW, int TS, typename S>
__global__ __launch_bounds__(NW * 64, MT <= 2 ? 4 : 2) void forward_split_kernel(Params P, PlanSet alts, const unsigned* __restrict__ sel,
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
    constexpr int TN = 32, WGS = NW * 64, NP = PT::NP;
    constexpr bool EARLY = MT == 4 || TS >= 8;          // weights requested before the step's samples: there are registers for it
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int sNonFinite, sRedo;
    typedef typename HaloCell<S>::Vec Cell;
    Cell* sIn = reinterpret_cast<Cell*>(smem_raw);
    const int lane = threadIdx.x & 63, wave = TS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int j = lane % TN, q = lane / TN;
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
        valid = tile_position<ND>(P, tg, wave / TS * TN + j, o, pos);
#pragma unroll
        for (int a = 0; a < ND; ++a) ib[a] = o[a] * P.stride[slot<ND>(a)] - P.pad[slot<ND>(a)];
    }

    typename MM::Acc acc[MT];
    const int ntg = (P.kV + 1) / 2;
    const unsigned mtiles = P.Mp / TN;
    const unsigned per_slab = (unsigned)ntg * mtiles * NP * 64;        // operands (16 bytes) of a slab
    const unsigned row = (unsigned)H.hext[2], plane = ND == 3 ? (unsigned)(H.hext[1] * H.hext[2]) : 0u;
    const unsigned a_lane = (unsigned)lane * 16;         // byte offset of this lane's operand
    const unsigned a_tg = mtiles * NP * 64;
    const int cg0 = g * P.Cg, cg1 = cg0 + P.Cg;

    // Ordered before the checks by the barriers of the first chunk.  sNonFinite stays set for the chunks that follow: cleared for each, it
    // could be cleared under a wavefront that has not read it yet by one that has no step in this chunk.
    if (threadIdx.x == 0) sRedo = sNonFinite = 0;
    // exact: the contraction on the float32 instructions, with the reference's treatment of non-finite
    // input next to the rim.
    auto work = [&](auto exact_tag) {
        constexpr bool exact = decltype(exact_tag)::value;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = acc_zero<float>();
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
                const int ngrp = (nch + FG - 1) / FG;
                const S* chan0 = in + ((size_t)n * P.C_in + cc0) * P.inV;      // workgroup-uniform
                // this wavefront's steps of the pass: [first, last) of the (tap pair, group) list
                const int steps = ntg * ngrp, first = TS > 1 ? steps * (wave % TS) / TS : 0, last = TS > 1 ? steps * (wave % TS + 1) / TS : steps;
                const float per = __builtin_amdgcn_rcpf((float)ngrp);                 // (floor((x + 0.5) / ngrp) for the few thousand steps of a pass)
                const int tg_first = TS > 1 ? __builtin_amdgcn_readfirstlane((int)(((float)first + 0.5f) * per)) : 0;
                const int tg_end = TS > 1 ? __builtin_amdgcn_readfirstlane((int)(((float)(last + ngrp - 1) + 0.5f) * per)) : ntg;
                float ofs[ND];
                load_pair_offsets<ND, S>(P, off_dg, min(tg_first, ntg - 1), q, pos, ofs, off == nullptr);
                __syncthreads();                                               // readers of the previous chunk are done
                if (stage_halo<ND, WGS, exact, S>(P, H, tg, chan0, nch, sIn)) sNonFinite = 1;
                __syncthreads();
                // Non-finite input in this halo or one before it (a non-finite sample always leads to the second pass): the
                // branch-free sampler reads the cell next to a collapsed corner with weight 0, and 0 * inf would
                // be NaN where the reference never touches that voxel
                // (deform3d/lib/deform_conv3d_cuda_kernel.cu:24-26).  Samples in the collapse zones (p <= 0 or
                // p >= size - 1 on some axis) are then taken from global memory with the reference's corner rule.
                const bool rim_far = exact && sNonFinite != 0;                 // uniform
                // (passes of four channels, where no more fit: every second one takes the upper half of its
                // group -- the operands from four elements further on, whose last four then meet zeros)
                const int upper = (cc0 - cb) & 4;
                const Elem* wchunk = Wq + ((size_t)chunk_slot<FG>(P.cpg, P.Cg, cc0 - upper) * per_slab * FG + (size_t)mchunk * MT * NP * 64 * FG + upper);
                int k0[ND];                            // kernel coordinates of the tap pair, counted up in scalar registers
#pragma unroll
                for (int a = 0; a < ND; ++a) k0[a] = 0;
                if constexpr (TS > 1) decode_tap<ND>(P, 2 * tg_first, k0);
                for (int tgi = tg_first; tgi < tg_end; ++tgi) {
                    int k1[ND];
#pragma unroll
                    for (int a = 0; a < ND; ++a) k1[a] = k0[a];
                    next_tap<ND>(P, k1);
                    SplitTap<ND> t;
                    split_geometry<ND>(P, H, tg, ib, q, k0, k1, ofs, valid && tgi * 2 + q < P.kV, rim_far, t);
                    // the next tap pair's offsets travel through this one's steps
                    load_pair_offsets<ND, S>(P, off_dg, min(tgi + 1, ntg - 1), q, pos, ofs, off == nullptr);
                    const bool any_far = __any(t.far); // rare: some sample of this wave reaches past the halo
                    const Elem* wp = wchunk + (size_t)tgi * a_tg * FG;
                    const int g0 = TS > 1 ? max(first - tgi * ngrp, 0) : 0, g1 = TS > 1 ? min(last - tgi * ngrp, ngrp) : ngrp;
                    if constexpr (TS > 1) wp += (size_t)g0 * per_slab * FG;
                    for (int grp = g0; grp < g1; ++grp) {
                        float val[FG];
                        Vec a8[MT][NP];
                        auto load_a = [&]() {
#pragma unroll
                            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                                for (int k = 0; k < NP; ++k) __builtin_memcpy(&a8[mt][k], reinterpret_cast<const char*>(wp) + (mt * NP + k) * 1024 + a_lane, 16);
                            __builtin_amdgcn_sched_barrier(0);      // all of them on their way while the operand is made
                        };
                        if constexpr (EARLY && !(exact && sizeof(S) == 4)) load_a();
                        // (corner reads ahead of what other wavefronts have to issue: 64 -> 64, 3x3x3, 4 x 16 x 56 x 56, 482 -> 476 us a call; elsewhere 0 to 0.5 %)
                        __builtin_amdgcn_s_setprio(1);
                        group_sum8<ND, S>(sIn, t.base, grp, nch, H.hstride, row, plane, t.cw, val);
                        __builtin_amdgcn_s_setprio(0);
                        if (__builtin_expect(any_far, 0)) far_values<ND, S>(P, t, chan0, grp * FG, nch, val);
                        if constexpr (!EARLY && !(exact && sizeof(S) == 4)) load_a();
                        if constexpr (!exact) {
                            Vec b8[NP];
                            PT::split(val, b8);
                            mma_parts<S, MT>(a8, b8, acc);
                        } else
                            mma_exact<S, MT>(P, W, g, mchunk * MT * TN + j, tgi * 2 + q, (size_t)(cc0 - cg0 + grp * FG), a8, val, t.near || t.far, nch - grp * FG, acc);
                        wp += (size_t)per_slab * FG;
                    }
                    next_tap<ND>(P, k1);
#pragma unroll
                    for (int a = 0; a < ND; ++a) k0[a] = k1[a];
                }
            }
        }
    };
    work(std::false_type{});
    if (valid && !results_stand<MT, S>(acc)) sRedo = 1;
    __syncthreads();
    if (__builtin_expect(sRedo, 0)) work(std::true_type{});
    if constexpr (TS >= 8) {
        // the sums of a position's TS wavefronts, [wavefront of the position][position tile][register][lane]: each adds up
        // and writes a share of the registers
        constexpr int NR = MT * MM::NACC, RW = NR / TS, PTS = NW / TS;
        __syncthreads();
        float* sum = reinterpret_cast<float*>(smem_raw);
        const int part_of = wave % TS, tile = wave / TS;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < MM::NACC; ++r) sum[((part_of * PTS + tile) * NR + mt * MM::NACC + r) * 64 + lane] = acc[mt][r];
        __syncthreads();
        const size_t at = (size_t)n * P.C_out * P.outV + pos;
#pragma unroll
        for (int x = 0; x < RW; ++x) {
            const int r = part_of * RW + x;                             // uniform
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < TS; ++k) v += sum[((k * PTS + tile) * NR + r) * 64 + lane];
            const int m = (mchunk * MT + r / MM::NACC) * TN + MM::row(r % MM::NACC, 0) + q * 4;
            if (valid && m < P.M) {
                const size_t to = at + ((size_t)g * P.M + m) * P.outV;
                if (U.split) part[(size_t)U.cz * P.N * P.C_out * P.outV + to] = v;      // (the bias is added when the parts are joined)
                else out[to] = Store<S>::st(bias ? v + Store<S>::ld(bias[g * P.M + m]) : v);
            }
        }
        return;
    } else if constexpr (TS > 1) {
        // the sums of a position's TS wavefronts, added in their order: [TS - 1][position tile][register][lane]
        __syncthreads();
        float* sum = reinterpret_cast<float*>(smem_raw);
        const int part_of = wave % TS, tile = wave / TS;
        if (part_of) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < MM::NACC; ++r) sum[((((part_of - 1) * (NW / TS) + tile) * MT + mt) * MM::NACC + r) * 64 + lane] = acc[mt][r];
        }
        __syncthreads();
        if (part_of) return;
        for (int k = 0; k < TS - 1; ++k)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int r = 0; r < MM::NACC; ++r) acc[mt][r] += sum[(((k * (NW / TS) + tile) * MT + mt) * MM::NACC + r) * 64 + lane];
    }

    if (U.split && whole > 0) {
        // partial sums of a unit of the last round: [split workgroup][MT * TN rows][NW * TN positions]
        constexpr int NP_ = NW / TS * TN;
        float* dst = part + (size_t)U.pslot * (MT * TN) * NP_ + q * 4 * NP_ + wave / TS * TN + j;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < MM::NACC; ++r) dst[(mt * TN + MM::row(r, 0)) * NP_] = acc[mt][r];
        return;
    }
    if (!valid) return;
    // unsplit: the output with bias; every unit split: a partial output tensor per cz, the bias is added when they are joined
    const size_t sample = (size_t)n * P.C_out * P.outV;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m0 = (mchunk * MT + mt) * TN;
        if (U.split) store_tile<float, S>(P, part + (size_t)U.cz * P.N * P.C_out * P.outV + sample, nullptr, g, m0, q, pos, acc[mt]);
        else store_tile<S, S>(P, out + sample, bias, g, m0, q, pos, acc[mt]);
    }
}

}  // namespace dcn
