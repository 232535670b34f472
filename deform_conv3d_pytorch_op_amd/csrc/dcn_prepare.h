// Everything a backward pass needs before its main kernels, in one launch.  The jobs are independent of
// each other -- weights packed in operand order, bounds of the weights, the choice of the halo plan,
// cleared gradients, channels-last copies with the sums of grad_output for grad_bias -- and each is a
// few microseconds of work: as launches of their own they cost a small layer more than the kernels they prepare
// (2 x 8 x 16 x 16 float64: eight launches of 1 to 6 us with gaps of 5 to 17 us between them).
// Large layers are bound by the copies: 64 -> 64 channels, 3-D, 4 x 16 x 56 x 56 float32, 411 MB in 100 us (4.1 TB/s; a plain
// copy reaches 5.1); 256 -> 256, 2-D, 8 x 56 x 56: 46 us; 128 -> 128, 3-D, 2 x 16 x 112 x 112 -> 56 x 56: 871 MB in 197.
#pragma once
#include "dcn_backward_fused.h"
#include "dcn_backward_weight_split.h"

namespace dcn {

enum PrepKind { PREP_PACK, PREP_FUSED_PACK, PREP_GOUT, PREP_PLAN, PREP_BOUNDS, PREP_ZERO, PREP_ROWS, PREP_LAST };
struct PrepJob {
    int kind, variant;          // PACK, FUSED_PACK: channels per chunk; PACK: + 1 for the wide row order
    unsigned first;             // first block; the job's blocks reach to the next job's first
    const void* src;
    void* dst;
    void* sums;                 // LAST: partial sums [C][strips of all samples], or null
    size_t n;                   // ZERO: 4-byte words
    int C;                      // LAST: channels, voxels, samples
    unsigned V;
    int N;
};
constexpr int MAX_PREP = 12;
struct PrepJobs {
    PrepJob job[MAX_PREP];
    int n;
};
constexpr unsigned LAST_STRIP = 256;       // voxels of a LAST block
__host__ __device__ inline unsigned last_strips(unsigned V) { return (V + LAST_STRIP - 1) / LAST_STRIP; }

// max |w| and the largest norm over the output channels of a group of an (input channel, tap) column:
// |grad column| <= that norm times the norm of grad_output over the output channels at the position
// (Cauchy-Schwarz).  Every block leaves the maxima of its columns as bit patterns, of which NaN is the
// largest; the readers take the maximum over the blocks (weight_bound).  Where the squares of a column may have underflowed (a sum below
// 2^-100) they are those of 2^96 times its values.
constexpr int BOUND_BLOCKS = 64;
template <typename S>
__device__ inline void prep_bounds(const Params& P, const S* __restrict__ w, float* __restrict__ out, unsigned block) {
    // 64 neighbouring columns of one group x 4 slices of its rows
    __shared__ float part[2][4][64];
    __shared__ unsigned amax[4];
    const int cx = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const size_t cols = (size_t)P.Cg * P.kV, tiles = (cols + 63) / 64;
    unsigned am = 0u, nm = 0u;
    for (size_t tile = block; tile < tiles * P.G; tile += BOUND_BLOCKS) {
        const size_t g = tile / tiles, col = tile % tiles * 64 + cx;
        float ss = 0.f, st = 0.f;
        if (col < cols) {
            const S* p = w + g * P.M * cols + col;
#pragma unroll 8
            for (int r = sl; r < P.M; r += 4) {
                const float v = offset_value(p[(size_t)r * cols]);
                ss += v * v;
                st += (v * 0x1p96f) * (v * 0x1p96f);
                am = max(am, __float_as_uint(fabsf(v)));
            }
        }
        part[0][sl][cx] = ss;
        part[1][sl][cx] = st;
        __syncthreads();
        ss = (part[0][0][cx] + part[0][1][cx]) + (part[0][2][cx] + part[0][3][cx]);
        st = (part[1][0][cx] + part[1][1][cx]) + (part[1][2][cx] + part[1][3][cx]);
        nm = max(nm, __float_as_uint(fabsf(ss < 0x1p-100f ? sqrtf(st) * 0x1p-96f : sqrtf(ss))));      // (false for NaN)
        __syncthreads();
    }
    for (int sh = 1; sh < 64; sh <<= 1) {
        am = max(am, (unsigned)__shfl_xor((int)am, sh));
        nm = max(nm, (unsigned)__shfl_xor((int)nm, sh));
    }
    if (cx == 0) amax[sl] = am;
    __syncthreads();
    if (threadIdx.x == 0) {
        out[2 * block] = __uint_as_float(max(max(amax[0], amax[1]), max(amax[2], amax[3])));
        out[2 * block + 1] = __uint_as_float(nm);
    }
}

// [C][V] -> [V][C] of one strip of voxels and 32 channels, 32 x 32 tiles through LDS, and the strip's sums
template <typename T, typename S>
__device__ inline void prep_channels_last(const PrepJob& job, unsigned block) {
    __shared__ S tile[32][33];
    const unsigned strips = last_strips(job.V), ctiles = ((unsigned)job.C + 31) / 32;
    const unsigned strip = block % strips, c0 = (block / strips) % ctiles * 32, n = block / strips / ctiles;
    const size_t base = (size_t)n * job.C * job.V;
    const S* src = static_cast<const S*>(job.src) + base;
    S* dst = static_cast<S*>(job.dst) + base;
    const unsigned tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    T sum[4] = {0, 0, 0, 0};
    // The next tile's values are on their way while this one is written; clamped, so that no load is masked.  (The launch was bounded
    // by the round trips to memory; us, a tile at a time -> so: 128 -> 128 channels in 3-D as above 244 -> 197, 64 -> 64 127 -> 100,
    // 256 -> 256 57 -> 46; a plain convolution of 25 088 positions 20 -> 12.  Tiles of 64 voxels are no faster.)
    S x[4];
    auto load = [&](unsigned v0) {
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) x[k] = src[(size_t)min(c0 + ty + 8 * k, (unsigned)job.C - 1) * job.V + min(v0 + tx, job.V - 1)];
    };
    const unsigned end = min((strip + 1) * LAST_STRIP, job.V);
    load(strip * LAST_STRIP);
    for (unsigned v0 = strip * LAST_STRIP; v0 < end; v0 += 32) {
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
            tile[ty + 8 * k][tx] = x[k];
            if (v0 + tx < job.V) sum[k] += (T)Store<S>::ld(x[k]);
        }
        __syncthreads();
        load(v0 + 32);
#pragma unroll
        for (unsigned k = 0; k < 4; ++k) {
            const unsigned v = v0 + ty + 8 * k, c = c0 + tx;
            if (c < (unsigned)job.C && v < job.V) dst[(size_t)v * job.C + c] = tile[tx][ty + 8 * k];
        }
        __syncthreads();
    }
    if (job.sums) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int sh = 1; sh < 32; sh <<= 1) sum[k] += __shfl_xor(sum[k], sh);
            const unsigned c = c0 + ty + 8 * k;
            if (tx == 0 && c < (unsigned)job.C) static_cast<T*>(job.sums)[(size_t)c * strips * job.N + n * strips + strip] = sum[k];
        }
    }
}

// grad_output in the operand order of backward_weight_split_kernel, and its sums: 32 channels of a strip, 64 positions at a
// time through LDS, then eight positions of one channel to a thread.
template <typename S>
__device__ inline void prep_rows(const PrepJob& job, unsigned block) {
    using PT = Parts<S>;
    __shared__ S tile[32][sizeof(S) == 4 ? 65 : 66];
    const unsigned strips = last_strips(job.V), ctiles = ((unsigned)job.C + 31) / 32;
    const unsigned strip = block % strips, c0 = (block / strips) % ctiles * 32, n = block / strips / ctiles;
    const S* src = static_cast<const S*>(job.src) + (size_t)n * job.C * job.V;
    const unsigned steps = row_steps(job.V), tx = threadIdx.x & 63, ty = threadIdx.x >> 6, c = c0 + (threadIdx.x & 31), oct = threadIdx.x >> 5;
    typename PT::Vec* dst = static_cast<typename PT::Vec*>(job.dst) + (size_t)n * steps * PT::NP * 2 * job.C;
    float sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    S x[8];                                             // (as in prep_channels_last)
    auto load = [&](unsigned v0) {
#pragma unroll
        for (unsigned k = 0; k < 8; ++k) x[k] = src[(size_t)min(c0 + ty + 4 * k, (unsigned)job.C - 1) * job.V + min(v0 + tx, job.V - 1)];
    };
    const unsigned end = min((strip + 1) * LAST_STRIP, job.V);
    load(strip * LAST_STRIP);
    for (unsigned v0 = strip * LAST_STRIP; v0 < end; v0 += 64) {
#pragma unroll
        for (unsigned k = 0; k < 8; ++k) {
            if (v0 + tx >= job.V) x[k] = S();
            tile[ty + 4 * k][tx] = x[k];
            sum[k] += Store<S>::ld(x[k]);
        }
        __syncthreads();
        load(v0 + 64);
        const unsigned step = (v0 >> 4) + (oct >> 1);
        if (c < (unsigned)job.C && step < steps) {
            typename PT::Vec p8[PT::NP];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                typename PT::Elem p[PT::NP];
                PT::split1(tile[threadIdx.x & 31][oct * 8 + e], p);
#pragma unroll
                for (int x = 0; x < PT::NP; ++x) p8[x][e] = p[x];
            }
#pragma unroll
            for (int x = 0; x < PT::NP; ++x) dst[((size_t)(step * 2 + (oct & 1)) * PT::NP + x) * job.C + c] = p8[x];
        }
        __syncthreads();
    }
    if (job.sums) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
#pragma unroll
            for (int sh = 1; sh < 64; sh <<= 1) sum[k] += __shfl_xor(sum[k], sh);
            const unsigned ch = c0 + ty + 4 * k;
            if (tx == 0 && ch < (unsigned)job.C) static_cast<float*>(job.sums)[(size_t)ch * strips * job.N + n * strips + strip] = sum[k];
        }
    }
}

template <typename T, typename S>
__global__ __launch_bounds__(256) void backward_prepare_kernel(Params P, PlanChoice pc, PrepJobs jobs, const S* __restrict__ W,
                                                               const S* __restrict__ off, size_t n_off) {
    touch_arguments<sizeof(Params) + sizeof(PlanChoice) + sizeof(PrepJobs) + 16>();
    // this block's job (selected field by field from constant argument offsets: a dynamic index would
    // put the whole list into scratch memory)
    PrepJob job = jobs.job[0];
    unsigned next = jobs.n > 1 ? jobs.job[1].first : gridDim.x;
#pragma unroll
    for (int k = 1; k < MAX_PREP; ++k)
        if (k < jobs.n && blockIdx.x >= jobs.job[k].first) {               // uniform
            job = jobs.job[k];
            next = k + 1 < MAX_PREP && k + 1 < jobs.n ? jobs.job[k + 1 < MAX_PREP ? k + 1 : k].first : gridDim.x;
        }
    const unsigned block = blockIdx.x - job.first, blocks = next - job.first;
    switch (job.kind) {
        case PREP_PACK: {
            S* dst = static_cast<S*>(job.dst);
            if (job.variant == 16) { if constexpr (sizeof(T) == 4) pack_backward_weight<T, 16, false, S>(P, W, dst, block, blocks); }
            else if (job.variant == 9) { if constexpr (sizeof(T) == 4) pack_backward_weight<T, 8, true, S>(P, W, dst, block, blocks); }
            else if (job.variant == 8) pack_backward_weight<T, 8, false, S>(P, W, dst, block, blocks);
            else pack_backward_weight<T, 4, false, S>(P, W, dst, block, blocks);
            break;
        }
        case PREP_FUSED_PACK: {
            if constexpr (sizeof(T) == 4) {
                typename Parts<S>::Vec* dst = static_cast<typename Parts<S>::Vec*>(job.dst);
                if (job.variant == 16) pack_fused_weight<16, S>(P, W, dst, block, blocks);
                else if (job.variant == 8) pack_fused_weight<8, S>(P, W, dst, block, blocks);
                else pack_fused_weight<4, S>(P, W, dst, block, blocks);
            }
            break;
        }
        case PREP_GOUT: {
            if constexpr (sizeof(T) == 4)
                split_grad_output<S>(P, static_cast<const S*>(job.src), static_cast<typename Parts<S>::Vec*>(job.dst), block, blocks);
            break;
        }
        case PREP_PLAN: choose_plan(pc, off, n_off); break;
        case PREP_BOUNDS: prep_bounds<S>(P, W, static_cast<float*>(job.dst), block); break;
        case PREP_ZERO: {
            // 16 bytes per store; the first and last words of an unaligned range one by one
            unsigned* p = static_cast<unsigned*>(job.dst);
            typedef unsigned U4 __attribute__((ext_vector_type(4)));
            const size_t head = min((size_t)((16 - ((size_t)p & 15)) & 15) / 4, job.n), quads = (job.n - head) / 4;
            U4* q = reinterpret_cast<U4*>(p + head);
            for (size_t i = (size_t)block * 256 + threadIdx.x; i < quads; i += (size_t)blocks * 256) q[i] = U4{0u, 0u, 0u, 0u};
            if (block == 0 && threadIdx.x < 8) {
                if (threadIdx.x < head) p[threadIdx.x] = 0u;
                const size_t at = head + quads * 4 + threadIdx.x;
                if (at < job.n) p[at] = 0u;
            }
            break;
        }
        case PREP_ROWS:
            if constexpr (sizeof(S) <= 4) prep_rows<S>(job, block);
            break;
        default: prep_channels_last<T, S>(job, block); break;
    }
}

// The list of jobs as the host puts it together.
struct Prep {
    PrepJobs jobs;
    unsigned blocks = 0;
    const float* octets = nullptr;              // where a 16-bit layer's grad_input was collected, if in octets (see dcn_backward_fused.h)
    bool full = false;                          // a job too many was added: launch_prepare then refuses
    Prep() { jobs.n = 0; }
    PrepJob& add(int kind, unsigned nblocks) {
        if (jobs.n == MAX_PREP) {
            full = true;
            return spare;
        }
        PrepJob& j = jobs.job[jobs.n++];
        j = PrepJob{kind, 0, blocks, nullptr, nullptr, nullptr, 0, 0, 0, 0};
        blocks += nblocks;
        return j;
    }
    void zero(void* p, size_t bytes) {          // a whole number of 4-byte words
        const size_t b = (bytes / 16 + 1023) / 1024;
        PrepJob& j = add(PREP_ZERO, (unsigned)(b < 1 ? 1 : b > 4096 ? 4096 : b));
        j.dst = p;
        j.n = bytes / 4;
    }
    void channels_last(const void* src, void* dst, int C, unsigned V, int N, void* sums) {
        PrepJob& j = add(PREP_LAST, last_strips(V) * (((unsigned)C + 31) / 32) * (unsigned)N);
        j.src = src; j.dst = dst; j.C = C; j.V = V; j.N = N; j.sums = sums;
    }
    void rows(const void* src, void* dst, int C, unsigned V, int N, void* sums) {
        PrepJob& j = add(PREP_ROWS, last_strips(V) * (((unsigned)C + 31) / 32) * (unsigned)N);
        j.src = src; j.dst = dst; j.C = C; j.V = V; j.N = N; j.sums = sums;
    }

private:
    PrepJob spare;
};

}  // namespace dcn
