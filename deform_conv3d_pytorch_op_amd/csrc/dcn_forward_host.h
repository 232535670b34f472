// Host side of the forward pass: plans and launches.
#pragma once
#include "dcn_host.h"
#include "dcn_forward.h"
#include "dcn_forward_shared.h"

namespace dcn {

constexpr size_t MAX_FORWARD_LDS = 160 * 1024 - 256;       // dynamic LDS of forward_split_kernel and forward_shared_kernel

// Which layers of 16-bit storage the halo kernels serve themselves: those whose halo fits at 256 positions to a
// block.  The kernels round every sample to the storage format, the float32 operator on widened tensors does not:
// the smaller blocks of few positions and of shared columns would fit more layers and give them less exact results
// (3x3x3, stride 2, dilation 2 in bfloat16: 2.3e-3 instead of 1.7e-3 from float64, 2-norm).
template <int ND>
bool forward16_native(const Params& P) {
    for (bool smallest : {false, true}) {
        Params Pt = P;
        if (plan_halo<float, ND>(Pt, MAX_FORWARD_LDS, default_margin(), 1 << 30, 2, WAVESH, smallest, FG, nullptr, 1, false)) return true;
    }
    return false;
}

// Channels per LDS pass, at most cchunk and a multiple of step, such that the passes of a group fall evenly on fsplit workgroups.
inline int even_chunk(const Params& P, int cchunk, int step, int fsplit) {
    for (int cc = cchunk; cc >= step; cc -= step) {
        int n = 0;
        for (int dg = 0; dg <= (P.Cg - 1) / P.cpg; ++dg) {
            const int len = (P.Cg < (dg + 1) * P.cpg ? P.Cg : (dg + 1) * P.cpg) - dg * P.cpg;
            n += (len + cc - 1) / cc;
        }
        if (n % fsplit == 0) return cc;
    }
    return cchunk;
}

// The plain convolution on a kernel of its own; *done says whether it took the layer.
inline int plain_forward(Params P, const float* in, const float* w, const float* bias, float* out, void* ws, size_t ws_bytes, hipStream_t s, bool* done) {
    *done = false;
    const PlainRows rows = plain_rows(P.M, P.kV);
    const int mw = rows.mw, rw = rows.rw;
    P.mchunks = rows.mchunks;
    P.Mp = rows.mchunks * mw * rw * 32;
    if (!plan_halo<float, 2>(P, (size_t)1 << 30, 0, 64, 1, PLAIN_COLS, false, FG, nullptr, 1, false)) return DCN_OK;
    const long long wgs = (long long)P.N * P.tiles * P.G * P.mchunks;
    P.cchunk = plain_channels(rows, wgs, P.cchunk, P.hvol, cu_count());
    const size_t lds = plain_lds(P.hvol, P.cchunk);
    if (lds > MAX_PLAIN_LDS || ws_bytes < split_weight_bytes<float>(P, P.Mp) || wgs > 0x7fffffffLL || !plain_conv()) return DCN_OK;
    if (plain_conv() != 2 && !plain_pays(rows, wgs, P.Cg, P.kV, P.hvol, cu_count())) return DCN_OK;
    *done = true;
    const unsigned items = (unsigned)chunk_candidates<FG>(P.cpg, P.Cg, P.C_in) * (unsigned)((P.kV + 1) / 2) * (unsigned)(P.Mp / 32), blocks = (items + 3) / 4;
    const PlanChoice none = {};
    hipLaunchKernelGGL(pack_split_weight_kernel<float>, dim3(blocks > 8192 ? 8192 : blocks), dim3(256), 0, s, P, w, static_cast<Parts<float>::Elem*>(ws), none,
                       static_cast<const float*>(nullptr), (size_t)0);
    if (int rc = check_launch("forward weight packing")) return rc;
    if (trace_plans())
        fprintf(stderr, "dcn plain convolution: %d wavefronts along the rows, %d row tiles each, %d channels at a time, grid %lld, LDS %zu\n", mw, rw, P.cchunk, wgs, lds);
    return launch_halo(plain_kernel(rows), "plain_conv_kernel", dim3((unsigned)wgs), PLAIN_COLS * mw * 64, lds, s, P, in, reinterpret_cast<const Parts<float>::Vec*>(ws), w, bias, out);
}

// S = T: the float32 / float64 operator.  S = Bf16 / Fp16 (T = float): the tensors are in that
// storage format and only the LDS-halo kernel serves them; where it cannot (halo too large, a layer
// that wants the input-channel split), *declined is set and nothing is launched: the caller then
// widens the tensors and runs the float32 operator.
template <typename T, int ND, typename S>
int forward(const Geometry& g, const S* in, const S* w, const S* off, const S* bias, S* out, void* ws,
            size_t ws_bytes, hipStream_t s, bool* declined, bool transposed) {
    constexpr bool S16 = !std::is_same<S, T>::value;
    constexpr bool MX = sizeof(T) == 4;                 // forward_split_kernel; float64: forward_quad_kernel
    constexpr size_t MAX_LDS = MX ? MAX_FORWARD_LDS : 144 * 1024;       // dynamic LDS of the only workgroup of a CU
    constexpr int CM = MX ? FG : FQ;                    // channels of a weight slab
    using WS = typename std::conditional<MX, S, float>::type;
    using WE = typename std::conditional<MX, typename Parts<WS>::Elem, S>::type;      // packed weight element
    auto slab_bytes = [](int kV, int Mp) {
        if constexpr (MX) return split_slab_elems<S>(kV, Mp) * sizeof(WE);
        else return forward_slab_elems<T>(kV, Mp) * sizeof(T);
    };
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (!in || !w || (!off && !MX) || !out) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    P.transposed = transposed ? 1 : 0;
    if (int rc = device_info(nullptr)) return rc;
    if constexpr (S16)
        if (!forward16_native<ND>(P)) { *declined = true; return DCN_OK; }
    if constexpr (ND == 2 && sizeof(S) == 4)
        if (!off) {
            bool done = false;
            if (int rc = plain_forward(P, in, w, bias, out, ws, ws ? ws_bytes : 0, s, &done)) return rc;
            if (done) return DCN_OK;
        }
    int MT, mchunks;
    fwd_weight_pad<T>(P.M, P.Cg, MT, mchunks, P.Mp, P.Cgp);
    P.mchunks = mchunks;
    if (!ws || (!S16 && ws_bytes < (size_t)P.G * P.kV * P.Mp * P.Cgp * sizeof(T))) return fail(DCN_E_WORKSPACE, "workspace too small");
    const int TN = Mma<T>::TN;
    // Too few position blocks to give every CU a workgroup.  First the input channels of a block are
    // split over up to FWD_MAX_SPLIT workgroups (each samples its own channels once; their partial
    // outputs are joined by a second kernel), as far as the workspace holds the partial outputs.
    // Then fewer row tiles per wavefront: more output-channel chunks, each sampling for itself.
    int fsplit = 1;
    const int mtiles_all = (P.M + TN - 1) / TN;
    // Which shape of the float32 / 16-bit kernels; times in us, float32 and 3x3 unless said otherwise.
    // Shared columns (forward_shared_kernel; units of 128 positions, MT = 4 or 8 row tiles): more than 64 output channels,
    // 2-D.  256 -> 256 channels, 8 x 56 x 56 positions: 239, and 277 where every wavefront samples for itself; 64 -> 512: 138 / 157;
    // in bfloat16 115 / 126 and 71 / 74.  3-D layers are not offered it: a block of 128 positions stages twice the halo
    // per position, 128 -> 128 channels at stride (1, 2, 2), 2 x 16 x 56 x 56 positions, 981 us and 1265 with shared columns (more output
    // channels or stride 1 would gain: -> 256 1807 / 1684, 64 -> 128 at stride 1, 2 x 16 x 28 x 28, 144 / 130).
    // Per 16 reduction slots and 32 positions a row tile costs its matrix instructions, and every chunk of row tiles
    // samples for itself (10 of the same unit): the cheaper of 4 and 8.  160 to 256 output channels, 8 samples: 238 with 8,
    // 289 with 4 row tiles.  (The number does not look at how far the
    // units fill the device: 3 samples of 64 -> 256, 84 units of 8 row tiles, take 73 where 168 of 4 take 48.)
    bool shared = MX && ND == 2 && mtiles_all > 2 && forward_shared();
    if (shared) {
        auto cost = [&](int rt) { const int mc = (mtiles_all + rt - 1) / rt; return mc * (rt * (S16 ? 1 : 6) + 10); };
        MT = mtiles_all > 4 && cost(8) <= cost(4) ? 8 : 4;
        P.mchunks = (mtiles_all + MT - 1) / MT;
    }
    // Few positions (`small`): forward_split_kernel in blocks of 64 positions, four wavefronts to a position, as long as
    // that gives a CU no more workgroups than it holds (two; one of four row tiles).  One sample, with / without:
    // 3x3x3, 64 -> 16 channels, 8 x 14 x 14 positions: 23 / 52; 124 layers of 16 to 256 channels: 0.85 of the time on average, at
    // worst 1.2 (2-D, 64 -> 64, 75 x 101 positions: 34 / 30).  Limits of half and of twice as many workgroups: the same
    // on average, single layers 0.7 to 0.8 times as fast.  Not for a single tap in 3-D: the halo of 64 positions costs more to
    // stage than it saves (128 -> 32 channels, 16 x 28 x 28: 42 with, 29 without).
    // And, of any number of positions, 3-D layers whose halo of 256 positions holds no eight channels (3x3x3 at stride 2 along every axis: 5733
    // voxels): they would take four at a time and leave half of the reduction slots empty.  Those of more than 64 output channels to a
    // group or at least 32 input channels, without / with, 3x3x3: 176 -> 151, 14 x 27 x 37 positions 1289 / 716; 64 -> 239, three samples of
    // 14 x 12 x 30 478 / 347; 64 -> 16, four of 17 x 18 x 19 252 / 216; 25 such layers 0.75 of the time on average, at worst 1.09 (16 -> 224 in two
    // groups, 75 / 81), and 0.6 with offsets that reach past the margins.  Fewer channels lose: 8 -> 24, 88 / 111.
    bool small = false;
    auto holds_eight = [&](bool smallest) {
        Params Pt = P;
        return plan_halo<T, ND>(Pt, MAX_LDS, default_margin(), 1 << 30, sizeof(S), WAVESH, smallest, FG, nullptr, 1, false);
    };
    const bool wide_halo = MX && !S16 && ND == 3 && (P.M > 64 || P.Cg >= 32) && !holds_eight(false) && !holds_eight(true);
    // Shared columns only where they can fill half of the device: with a workgroup for every 16 input channels in
    // float32, whose channels can be split, and without in 16-bit storage, whose cannot (256 -> 256 channels, 3x3, 2 x 28 x 28
    // positions in bfloat16: 16 units, 105 us shared and 60 with several wavefronts to a position).
    if (MX && shared) {
        Params Pt = P;
        if (plan_halo<T, ND>(Pt, MAX_LDS, default_margin(), 1 << 30, sizeof(S), SHARED_COLS, false, FG, nullptr, 1, false) &&
            (long long)Pt.N * Pt.tiles * P.G * P.mchunks * (!S16 && P.Cg >= 32 ? P.Cg / 16 : 1) * 2 < cu_count())
            shared = false;
    }
    if (MX && !shared && (ND == 2 || P.kV > 1) && forward_small() && forward_slots() == 0) {
        Params Pt = P;
        const int mt = mtiles_all > 2 ? 4 : mtiles_all, mc = (mtiles_all + mt - 1) / mt;
        if (plan_halo<T, ND>(Pt, MAX_LDS, default_margin(), 1 << 30, sizeof(S), 2, false, FG, nullptr, 1, false) &&
            (long long)Pt.N * Pt.tiles * P.G * mc <= (wide_halo ? 0x7fffffffLL : (mt == 4 ? 1 : 2) * cu_count())) {
            small = true;
            MT = mt;
            P.mchunks = mc;
        }
    }
    const size_t out_bytes = (size_t)P.N * P.C_out * P.outV * sizeof(T);
    const size_t wq_bound = align256(((size_t)chunk_slot<CM>(P.cpg, P.Cg, P.C_in - 1) + 1) * slab_bytes(P.kV, (mtiles_all + 7) / 8 * 8 * TN));
    // Fewer positions still (`tiny`, position tiles of a block: 1 or 2): sixteen wavefronts to 32 positions or eight each to 64,
    // and as many parts of the input channels as pay, while that is one workgroup to a CU.  By estimated time: 2.5 us for a pass,
    // 2.0 (3-D) or 0.8 for a wavefront's step, 0.4 for a thread's cell to stage, 5 for joining parts, 2 for sixteen wavefronts.  One sample,
    // float32, with / without: 2-D, 64 -> 64, 75 x 101: 20.4 / 33; 48 -> 64, 5x5, 70 x 76: 25 / 49; 3-D, 128 -> 32 at stride 1 2 2, 14 x 20 x 20:
    // 65 / 102; two samples of 32 -> 16, 15 x 18 x 18: 30 / 55; 70 layers of 8 to 256 channels and 150 to 16 000
    // positions, 2-D and 3-D, also in bfloat16: 0.85 of the time on average.  Only where the estimate falls by a fifth: of 60 layers
    // below 6e6 samples those taken for less of it are the slower ones (320 -> 16, 3x3 at stride 2, 27 x 25: 25.4 / 27.9; 3-D, 32 -> 49 in
    // deformable groups of 8, 9 x 13 x 14: 24.5 / 26.2; without the line 0.867 of the time on average, with it 0.862, at worst 1.005).
    int tiny = 0;
    if (small && MT <= 2 && forward_tiny()) {
        const size_t room = ws_bytes > wq_bound ? (ws_bytes - wq_bound < FWD_PARTIAL_CAP ? ws_bytes - wq_bound : FWD_PARTIAL_CAP) : 0;
        auto parts_fit = [&](int fs) {
            return fs == 1 || (!S16 && fs <= forward_split() && fs <= FWD_MAX_SPLIT && (size_t)P.N * P.outV < FWD_SPLIT_POSITIONS && (size_t)fs * out_bytes <= room && fs * FG <= P.Cg);
        };
        // the longest workgroup of fs to a block of t position tiles, ts wavefronts to a position
        auto estimate = [&](const Params& Pt, int t, int ts, int fs) {
            double load[FWD_MAX_SPLIT] = {0}, worst = 0;
            int k = 0;
            const int cch = fs > 1 ? even_chunk(P, Pt.cchunk, FG, fs) : Pt.cchunk;
            for (int dg = 0; dg <= (P.Cg - 1) / P.cpg; ++dg) {
                const int len = (P.Cg < (dg + 1) * P.cpg ? P.Cg : (dg + 1) * P.cpg) - dg * P.cpg;
                for (int c0 = 0; c0 < len; c0 += cch, ++k) {
                    const int n = len - c0 < cch ? len - c0 : cch, steps = (P.kV + 1) / 2 * ((n + FG - 1) / FG), cells = (n + HaloCell<WS>::CH - 1) / HaloCell<WS>::CH;
                    load[k % fs] += 2.5 + (ND == 3 ? 2.0 : 0.8) * ((steps + ts - 1) / ts) + 0.4 * cells * Pt.hvol / (t * ts * 64);
                }
            }
            for (int z = 0; z < fs; ++z) worst = load[z] > worst ? load[z] : worst;
            return worst + (fs > 1 ? 5 : 0) + (t * ts == 16 ? 2 : 0);
        };
        double best = 1e30;
        {   // four wavefronts to a position: as many parts as fit, below
            Params Pt = P;
            if (plan_halo<T, ND>(Pt, MAX_LDS / 2, default_margin(), 1 << 30, sizeof(S), 2, false, FG, nullptr, 1, false)) {
                int fs = 1;
                while (parts_fit(fs * 2) && (long long)Pt.N * Pt.tiles * P.G * P.mchunks * fs * 2 <= 2 * cu_count()) fs *= 2;
                best = estimate(Pt, 2, 4, fs);
            }
        }
        for (int t = 1; t <= 2; ++t) {
            Params Pt = P;
            const bool forced = forward_tiny() == t;
            if (forward_tiny() > 0 && !forced) continue;
            if (!plan_halo<T, ND>(Pt, MAX_LDS, default_margin(), 1 << 30, sizeof(S), t, true, FG, nullptr, 1, false)) continue;
            for (int fs = 1; parts_fit(fs) && ((long long)Pt.N * Pt.tiles * P.G * P.mchunks * fs <= cu_count() || (forced && fs == 1)); fs *= 2) {
                const double e = estimate(Pt, t, 16 / t, fs);
                if (e < (tiny ? best : 0.8 * best) || (forced && !tiny)) { best = e; tiny = t; fsplit = fs; }
            }
        }
    }
    const int nwp = shared ? SHARED_COLS : tiny ? tiny : small ? 2 : WAVESH;      // column tiles of a block
    {
        Params Pt = P;
        const bool tiled = plan_halo<T, ND>(Pt, MAX_LDS, default_margin(), 1 << 30, MX ? sizeof(S) : sizeof(T), nwp, false, FQ, nullptr, 1, !MX);
        const long long tiles = tiled ? (long long)Pt.N * Pt.tiles : (long long)P.N * ((P.outV + WAVES * TN - 1) / (WAVES * TN));
        // (eight row tiles per wavefront only pay when the grid is full anyway: measured slower than
        // four with twice the sampling)
        if (MT == 8 && !shared && (MX || tiles * P.G * P.mchunks < cu_count())) {
            MT = 4;
            P.mchunks = (mtiles_all + MT - 1) / MT;
        }
        // Parts of the input channels, as many as the device has room for, at least 16 channels each (8 where four wavefronts
        // share them; 4 or 16 there: 5 % slower, the same on average).  256 -> 16 channels, 28 x 28 positions: 44 unsplit, 22 split; 3x3x3,
        // 64 -> 16, 8 x 20 x 20: 71 / 37.  The join and a second workgroup on a CU cost more than short chains gain: 64 -> 64,
        // 112 x 112: 25 unsplit, 37 in two parts.
        if (!S16 && tiled && !tiny && forward_split() > 1 && (size_t)P.N * P.outV < FWD_SPLIT_POSITIONS && ws_bytes > wq_bound) {
            const size_t room = ws_bytes - wq_bound < FWD_PARTIAL_CAP ? ws_bytes - wq_bound : FWD_PARTIAL_CAP;
            while (fsplit * 2 <= FWD_MAX_SPLIT && fsplit * 2 <= forward_split() && tiles * P.G * P.mchunks * fsplit * 2 <= (small && MT < 4 ? 2 : 1) * cu_count() &&
                   (size_t)fsplit * 2 * out_bytes <= room && fsplit * 2 * (small ? 8 : 16) <= P.Cg)
                fsplit *= 2;
        }
        // Fewer row tiles, more chunks of them, while the grid fills less than half of the device (float64: less than all):
        // 3x3x3, 16 -> 128 channels, 16 x 40 x 40 positions: 58; limits of all or a quarter of the device: 72, 77.
        while (MT > 1 && !shared && !small && tiles * P.G * P.mchunks * fsplit < cu_count() / (MX ? 2 : 1)) {
            MT /= 2;
            P.mchunks = (mtiles_all + MT - 1) / MT;
        }
        P.Mp = P.mchunks * MT * TN;
    }
    // Halo kernel: a workgroup's input neighbourhood in LDS, several channels of a voxel side by side.  Few
    // accumulators (MT <= 2): one 1024-thread workgroup per CU with the whole LDS, if its larger halo
    // fits and leaves 8 channels per pass.  Otherwise 512 threads: two workgroups per CU when that
    // still leaves 8 channels per LDS pass, else one large one.  Returns the wavefronts per
    // workgroup, 0 when no halo of margin m fits.
    // channels per LDS pass: multiples of eight for forward_split_kernel, where they fit
    auto plan_shape = [&](Params& Ph, size_t budget, int m, int waves, bool smallest, const Div* blocks = nullptr) {
        if constexpr (MX)
            if (plan_halo<T, ND>(Ph, budget, m, 1 << 30, sizeof(S), waves, smallest, FG, blocks, 1, false)) return true;
        return !S16 && plan_halo<T, ND>(Ph, budget, m, MX ? 4 : 1 << 30, sizeof(T), waves, smallest, FQ, blocks, 1, !MX);
    };
    auto plan_for = [&](int m, Params& Ph) {
        Ph = P;
        int nw = 0;
        if (shared) {
            const size_t room = MAX_LDS - shared_column_bytes<typename std::conditional<MX, S, float>::type>();
            bool tiled = plan_halo<T, ND>(Ph, room, m, 1 << 30, sizeof(S), SHARED_COLS, false, FG, nullptr, 1, false);
            if (!tiled || Ph.cchunk < 16) {
                Params Ps = P;
                if (plan_halo<T, ND>(Ps, room, m, 1 << 30, sizeof(S), SHARED_COLS, true, FG, nullptr, 1, false) && (!tiled || Ps.cchunk > Ph.cchunk)) { Ph = Ps; tiled = true; }
            }
            return tiled && (long long)Ph.N * Ph.tiles * Ph.G * Ph.mchunks <= 0x7fffffffLL ? SHARED_COLS : 0;
        }
        if (small) {
            if (tiny) return plan_halo<T, ND>(Ph, MAX_LDS, m, 1 << 30, sizeof(S), tiny, true, FG, nullptr, 1, false) ? tiny : 0;
            // (half of the LDS: two workgroups share a CU)
            const bool tiled = plan_halo<T, ND>(Ph, MT == 4 ? MAX_LDS : MAX_LDS / 2, m, 1 << 30, sizeof(S), 2, false, FG, nullptr, 1, false) ||
                               plan_halo<T, ND>(Ph, MAX_LDS, m, 1 << 30, sizeof(S), 2, false, FG, nullptr, 1, false);
            return tiled ? 2 : 0;
        }
        // (the 3-D double instance of the 1024-thread shape does not fit its 128 registers.  float32: the two shapes
        // measure the same, 64 -> 32 and 64 channels in segments of 4 to 64, 2-D and 3-D: 0.98 to 1.02.)
        if (MT <= 2 && wide_forward() && !(sizeof(T) == 8 && ND == 3) && (!MX || wide_forward() == 2 || (P.cpg >= 16 && P.Cg >= 16))) {
            Params Pw = P;
            if (plan_shape(Pw, MAX_LDS, m, 16, false) && (long long)Pw.N * Pw.tiles * Pw.G * Pw.mchunks <= 0x7fffffffLL &&
                (wide_forward() == 2 || (Pw.cchunk >= 8 && (long long)Pw.N * Pw.tiles * Pw.G * Pw.mchunks >= cu_count()))) {
                Ph = Pw;
                nw = 16;
            }
        }
        if (!nw) {
            bool tiled = plan_shape(Ph, LDS_BUDGET, m, WAVESH, false);
            if ((!tiled || Ph.cchunk < 8) && LDS_BUDGET < MAX_LDS) tiled = plan_shape(Ph, MAX_LDS, m, WAVESH, false) || tiled;
            if (!tiled || Ph.cchunk < 8) {       // strided layers: the block shape with the smallest halo may hold 8 channels
                Params Ps = P;
                if (plan_shape(Ps, MAX_LDS, m, WAVESH, true) && (!tiled || Ps.cchunk > Ph.cchunk)) {
                    Ph = Ps;
                    tiled = true;
                }
            }
            if (tiled && (long long)Ph.N * Ph.tiles * Ph.G * Ph.mchunks <= 0x7fffffffLL) nw = WAVESH;
        }
        return nw;
    };
    {
        int margins[MAX_PLANS];
        int nmargins = plan_margins(ND, margins);
        if (!off && halo_margin() < 0) {       // samples at integer coordinates: their high corners are one voxel on
            nmargins = 1;
            margins[0] = 1;
        }
        Params plans[MAX_PLANS];
        int nw = plan_for(margins[0], plans[0]);
        if (shared && !nw) {       // (no halo of 128 positions holds eight channels)
            shared = false;
            MT = 4;
            P.mchunks = (mtiles_all + MT - 1) / MT;
            P.Mp = P.mchunks * MT * TN;
            nw = plan_for(margins[0], plans[0]);
        }
        if (small && !nw) return fail(DCN_E_LAUNCH, "no halo plan");      // (planned above)
        const size_t col_bytes = shared ? shared_column_bytes<typename std::conditional<MX, S, float>::type>() : 0;
        size_t wq_bytes;
        if constexpr (MX) wq_bytes = split_weight_bytes<S>(P, P.Mp);
        else wq_bytes = ((size_t)chunk_slot<CM>(P.cpg, P.Cg, P.C_in - 1) + 1) * slab_bytes(P.kV, P.Mp) + 256;
        auto halo_lds = [=](const Params& Ph) { return col_bytes + (size_t)Ph.cchunk * Ph.hstride * (MX ? sizeof(S) : sizeof(T)) + (MX ? 0 : (size_t)Ph.hvol * 4); };
        if (nw == 16 || ws_bytes < align256(wq_bytes) + (size_t)fsplit * out_bytes) fsplit = 1;
        if (nw && ws_bytes >= wq_bytes) {
            // channels per LDS pass such that every workgroup of a block gets the same number of passes
            auto even_passes = [&](Params& Ph) { Ph.cchunk = even_chunk(P, Ph.cchunk, Ph.cchunk % CM == 0 ? CM : FQ, fsplit); };
            if (fsplit > 1) even_passes(plans[0]);
            // Wider halos that one launch of the same kernel can serve as well (same workgroup shape and
            // position blocks); the choice among them is made on the device, see PlanChoice.  The
            // chosen index lives in the last 256 bytes of the workspace.
            PlanChoice pc = {};
            pc.nplans = 1;
            pc.nd = ND;
            pc.margin[0] = margins[0];
            pc.base[0] = 1.f;
            // How the time grows with the halo, and what samples beyond it cost, in times of a launch without any
            // (PlanChoice).  forward_split_kernel and forward_shared_kernel, offsets U[-r, r], us per margin (64 -> 64 channels,
            // 3x3x3, 4 x 16 x 28 x 28 positions; 256 -> 256, 3x3, 8 x 56 x 56):
            //   3-D, margins 2 / 3 / 4   r = 2: 161 / 169 / 177   r = 2.5: 376 / 169 / 177   r = 5: 688 / 543 / 378   r = 8: 924 / 808 / 683
            //   2-D, margins 2 / 4 / 6   r = 2: 238 / 250 / 262   r = 2.5: 336 / 250 / 262   r = 5: 380 / 349 / 262   r = 8: 430 / 408 / 374
            // A pass of four channels (3-D, where the wider halo holds no eight) leaves half of the reduction slots empty: 1.55
            // times the time.  float64: forward_quad_kernel walks the channels of a wavefront with such a sample once more.
            const float grow = MX ? (ND == 3 ? 0.1f : 0.12f) : ND == 3 ? 0.3f : 0.12f;
            pc.far_wave = MX ? (ND == 3 ? 0.6f : 0.4f) : ND == 3 ? 0.5f : 0.1f;
            pc.far_sample = MX ? (ND == 3 ? 1.3f : 0.4f) : ND == 3 ? 2.2f : 5.f;
            pc.far_steep = MX ? (ND == 3 ? 2.5f : 0.4f) : 0.f;
            const size_t used = align256(wq_bytes) + (fsplit > 1 ? (size_t)fsplit * out_bytes : 0);
            if (nmargins > 1 && ws_bytes >= used + 512) {
                // (within the LDS of the first plan, which fixes how many workgroups share a CU; all of it
                // when the grid gives a CU one workgroup at most)
                const long long wgs = (long long)plans[0].N * plans[0].tiles * plans[0].G * plans[0].mchunks * fsplit;
                size_t lds0 = halo_lds(plans[0]);
                // (... or its registers allow no more: 16 wavefronts of up to 128)
                if ((wgs <= cu_count() || shared || (MX && nw == 16)) && lds0 < MAX_LDS) lds0 = MAX_LDS;
                if (small && wgs > cu_count() && lds0 < MAX_LDS / 2) lds0 = MAX_LDS / 2;
                for (int k = 1; k < nmargins; ++k) {
                    Params& Pk = plans[pc.nplans];
                    Pk = P;
                    if (shared || small ? !plan_halo<T, ND>(Pk, lds0 - col_bytes, margins[k], 1 << 30, sizeof(S), nw, false, FG, plans[0].tdim, 1, false)
                               : !plan_shape(Pk, lds0, margins[k], nw, false, plans[0].tdim)) continue;
                    if (!same_blocks(Pk, plans[0]) || Pk.hvol > 3 * plans[0].hvol) continue;
                    if (fsplit > 1) even_passes(Pk);
                    pc.margin[pc.nplans] = margins[k];
                    pc.base[pc.nplans] = 1.f + grow * ((float)Pk.hvol / (float)plans[0].hvol - 1.f);
                    if (MX && Pk.cchunk % FG && plans[0].cchunk % FG == 0) pc.base[pc.nplans] *= 1.55f;
                    ++pc.nplans;
                }
                if (pc.nplans > 1) pc.sel = reinterpret_cast<unsigned*>(static_cast<char*>(ws) + (ws_bytes - 256) / 256 * 256);
            }
            for (int k = pc.nplans; k < MAX_PLANS; ++k) {
                plans[k] = plans[0];
                pc.margin[k] = pc.margin[pc.nplans - 1];
                pc.base[k] = 1e30f;
            }
            PlanSet alts;
            for (int k = 1; k < MAX_PLANS; ++k) alts.alt[k - 1] = halo_plan_of(plans[k]);
            alts.mask = (1u << pc.nplans) - 1;
            {
                size_t total = (size_t)chunk_candidates<CM>(P.cpg, P.Cg, P.C_in);
                if constexpr (MX) total *= (size_t)((P.kV + 1) / 2) * P.Mp * 2;          // one thread per operand of a lane
                else total *= forward_slab_elems<T>(P.kV, P.Mp);
                const unsigned blocks = (unsigned)((total + 255) / 256 > 8192 ? 8192 : (total + 255) / 256);
                const size_t n_off = (size_t)P.N * P.DG * P.kV * ND * P.outV;
                const dim3 pgrid(blocks + (pc.sel ? 1 : 0));
                if constexpr (MX) hipLaunchKernelGGL(pack_split_weight_kernel<S>, pgrid, dim3(256), 0, s, plans[0], w, static_cast<WE*>(ws), pc, off, n_off);
                else hipLaunchKernelGGL(pack_forward_weight_kernel<T>, pgrid, dim3(256), 0, s, plans[0], w, static_cast<T*>(ws), pc, off, n_off);
                if (int rc = check_launch("forward weight packing")) return rc;
            }
            // a grid of at most one workgroup per CU: sixteen wavefronts to its 256 positions, two to a position
            // (224 x 224 positions: 256 -> 16 channels 121, and 137 with one wavefront to a position; 16 -> 64: 28 / 25)
            const bool pairs = MX && !small && !shared && nw == WAVESH && MT <= 2 && P.kV > 1 && forward_small() && forward_slots() == 0 &&
                               (long long)plans[0].N * plans[0].tiles * plans[0].G * plans[0].mchunks * fsplit <= cu_count();
            // (the sums of the wavefronts that share positions)
            size_t lds = tiny ? (size_t)16 * MT * 4096 : small ? (size_t)3 * 2 * MT * 4096 : pairs ? (size_t)WAVESH * MT * 4096 : 0;
            for (int k = 0; k < pc.nplans; ++k) {
                const size_t l = halo_lds(plans[k]);
                if (l > lds) lds = l;
            }
            const Params& Ph = plans[0];
            using KernMx = void (*)(Params, PlanSet, const unsigned*, const S*, const S*, const WE*, const S*, const S*, S*, T*, Div, unsigned, TailSplit);
            using KernQuad = void (*)(Params, PlanSet, const unsigned*, const S*, const S*, const WE*, const S*, S*, T*, Div, unsigned, TailSplit);
            typename std::conditional<MX, KernMx, KernQuad>::type kern = nullptr;
            if constexpr (MX) {
                if (pairs) kern = MT == 1 ? forward_split_kernel<ND, 1, 16, 2, S> : forward_split_kernel<ND, 2, 16, 2, S>;
                else if (tiny == 1) kern = MT == 1 ? forward_split_kernel<ND, 1, 16, 16, S> : forward_split_kernel<ND, 2, 16, 16, S>;
                else if (tiny == 2) kern = MT == 1 ? forward_split_kernel<ND, 1, 16, 8, S> : forward_split_kernel<ND, 2, 16, 8, S>;
                else if (small) kern = MT == 1 ? forward_split_kernel<ND, 1, 8, 4, S> : MT == 2 ? forward_split_kernel<ND, 2, 8, 4, S> : forward_split_kernel<ND, 4, 8, 4, S>;
                else if (shared) { if constexpr (ND == 2) kern = MT == 8 ? forward_shared_kernel<ND, 8, S> : forward_shared_kernel<ND, 4, S>; }
                else if (nw == 16) kern = MT == 1 ? forward_split_kernel<ND, 1, 16, 1, S> : forward_split_kernel<ND, 2, 16, 1, S>;
                else kern = MT == 1 ? forward_split_kernel<ND, 1, WAVESH, 1, S> : MT == 2 ? forward_split_kernel<ND, 2, WAVESH, 1, S>
                                                                             : forward_split_kernel<ND, 4, WAVESH, 1, S>;
            } else {
                if (nw == 16) kern = MT == 1 ? forward_quad_kernel<T, ND, 1, 16> : forward_quad_kernel<T, ND, 2, 16>;
                else kern = MT == 1 ? forward_quad_kernel<T, ND, 1, WAVESH> : MT == 2 ? forward_quad_kernel<T, ND, 2, WAVESH>
                          : MT == 4 ? forward_quad_kernel<T, ND, 4, WAVESH> : forward_quad_kernel<T, ND, 8, WAVESH>;
            }
            T* part = reinterpret_cast<T*>(static_cast<char*>(ws) + align256(wq_bytes));      // partial sums, in the arithmetic type
            // A grid that ends in a partly filled round of workgroups: the units of that round, last in
            // the launch, are split over several workgroups each (every tsplit-th channel pass), so that
            // the round fills the device; forward_join_tail_kernel adds their partial sums.  Either all
            // of them tsplit ways, or -- when that leaves the last of the resulting short rounds partly
            // empty -- as many of them tsplit + 1 ways as make the workgroup count a whole number of
            // rounds (TailSplit: the units split tsplit ways come first, so that the longer workgroups
            // start first).  Cost of a workgroup: per channel pass one part for the tap geometry and one
            // per four channels, plus 5 % of a unit for its fixed part (halo table, offsets, output).
            const long long units = (long long)Ph.N * Ph.tiles * Ph.G * Ph.mchunks;
            int tsplit = 1;
            long long whole = 0;
            TailSplit ts = {0u, Div(0), 0};
            if (fsplit == 1 && !tiny && forward_tail_split()) {
                const long long slots = forward_slots() ? forward_slots() : resident_workgroups(reinterpret_cast<const void*>(kern), (pairs || tiny ? 16 : shared || small ? 8 : nw) * 64, lds);
                const long long rest = units % slots;
                // tap geometry of a pass, in units of four channels' sampling and contraction (35 layers of 32 to 128
                // channels whose last round is partly filled: 0.2 and 0.9 choose splits of the same time, no split takes 1.09 times as long)
                constexpr double GEO = 0.45;
                // cost of the longest workgroup when the passes of a unit (cch channels each) are dealt to cs workgroups
                auto wg_cost = [&](int cs, int cch, int* npasses) {
                    double load[64] = {0};
                    int k = 0;
                    for (int dg = 0; dg <= (P.Cg - 1) / P.cpg; ++dg) {
                        const int len = (P.Cg < (dg + 1) * P.cpg ? P.Cg : (dg + 1) * P.cpg) - dg * P.cpg;
                        for (int c0 = 0; c0 < len; c0 += cch, ++k) load[k % cs] += GEO + (double)(((len - c0 < cch ? len - c0 : cch) + FQ - 1) / FQ);
                    }
                    if (npasses) *npasses = k;
                    double worst = 0;
                    for (int z = 0; z < cs; ++z) worst = load[z] > worst ? load[z] : worst;
                    return worst;
                };
                int passes = 0;                 // channel passes of a unit under the first plan
                const double unit_cost = wg_cost(1, Ph.cchunk, &passes);
                const size_t end = pc.sel ? (ws_bytes - 256) / 256 * 256 : ws_bytes;
                const size_t room = end > align256(wq_bytes) ? end - align256(wq_bytes) : 0;
                const size_t per_wg = (size_t)MT * TN * nw * TN * sizeof(T);
                if (units > slots && rest) {
                    double best = 0.9;          // of the time of an unsplit last round; a tenth must be gained
                    for (int cs = 2; cs <= 8 && cs <= passes; ++cs) {
                        if (forward_tail_split() > 1 && cs != forward_tail_split()) continue;
                        const long long rounds = (rest * cs + slots - 1) / slots;
                        const double ta = wg_cost(cs, Ph.cchunk, nullptr) / unit_cost + 0.05;
                        {
                            const double t = (double)rounds * ta;
                            const size_t bytes = (size_t)rest * cs * per_wg;
                            if ((t < best || forward_tail_split() > 1) && bytes <= room && bytes <= FWD_PARTIAL_CAP) {
                                best = t; tsplit = cs; ts = TailSplit{0u, Div(0), 0};
                            }
                        }
                        // two runs: nb units cs + 1 ways, the others cs ways, rounds * slots workgroups in all;
                        // the cs-way workgroups must fit the first round
                        const long long nb = rounds * slots - rest * cs;
                        if (!forward_tail_two_runs() || cs + 1 > 8 || nb <= 0 || nb >= rest || (rest - nb) * cs > slots) continue;
                        double tb = 1e30;
                        int cchb = Ph.cchunk;
                        const int step = Ph.cchunk % CM == 0 ? CM : FQ;
                        for (int cch = Ph.cchunk; cch >= step; cch -= step) {
                            int np = 0;
                            const double c = wg_cost(cs + 1, cch, &np) / unit_cost + 0.05;
                            if (np >= cs + 1 && c < tb) { tb = c; cchb = cch; }
                        }
                        const double t = ta + (double)(rounds - 1) * tb;
                        const size_t bytes = (size_t)(rounds * slots) * per_wg;
                        if (t < best && bytes <= room && bytes <= FWD_PARTIAL_CAP) {
                            best = t; tsplit = cs; ts = TailSplit{(unsigned)(rest - nb), Div((int)cs + 1), cchb};
                        }
                    }
                    if (tsplit > 1) whole = units - rest;
                }
            }
            const long long wgs = tsplit > 1 ? whole + (ts.splitB ? (long long)ts.unitsA * tsplit + (units - whole - ts.unitsA) * ts.splitB : (units - whole) * tsplit)
                                             : units * fsplit;
            if (wgs > 0x7fffffffLL) return fail(DCN_E_ARGUMENT, "too many workgroups for one launch");
            const dim3 grid((unsigned)wgs);
            if (trace_plans()) {
                fprintf(stderr, "dcn forward: %d position tiles, %d wavefronts, MT %d, grid %u (%lld unsplit, rest x %d), LDS %zu, every unit split x %d\n", nw,
                        pairs || tiny ? 16 : shared || small ? 8 : nw, MT, grid.x, tsplit > 1 ? whole : 0LL, tsplit, lds, fsplit);
                if (ts.splitB) fprintf(stderr, "  of the rest: %u units x %d, the others x %d with %d channels per pass\n", ts.unitsA, tsplit, (int)ts.splitB, ts.cchB);
                for (int k = 0; k < pc.nplans; ++k)
                    fprintf(stderr, "  plan %d: margin %d, halo %d x %d x %d, %d channels per pass, base cost %.3f\n", k, pc.margin[k],
                            plans[k].hext[0], plans[k].hext[1], plans[k].hext[2], plans[k].cchunk, pc.base[k]);
            }
            const unsigned* sel = pc.sel;
            const int threads = (pairs || tiny ? 16 : shared || small ? 8 : nw) * 64, splits = tsplit > 1 ? tsplit : fsplit;
            int rc;
            if constexpr (MX) rc = launch_halo(kern, "forward halo kernel", grid, threads, lds, s, Ph, alts, sel, in, off, (const WE*)ws, w, bias, out, part, Div(splits), (unsigned)whole, ts);
            else rc = launch_halo(kern, "forward halo kernel", grid, threads, lds, s, Ph, alts, sel, in, off, (const WE*)ws, bias, out, part, Div(splits), (unsigned)whole, ts);
            if (rc) return rc;
            if (fsplit == 1 && tsplit == 1) return DCN_OK;
            if (tsplit > 1) {
                using Join = void (*)(Params, PlanSet, const unsigned*, const T*, const S*, S*, int, unsigned, TailSplit);
                Join join;
                if (small) join = MT == 1 ? forward_join_tail_kernel<T, ND, 1, 2, S> : MT == 2 ? forward_join_tail_kernel<T, ND, 2, 2, S> : forward_join_tail_kernel<T, ND, 4, 2, S>;
                else if (shared) join = MT == 8 ? forward_join_tail_kernel<T, ND, 8, SHARED_COLS, S> : forward_join_tail_kernel<T, ND, 4, SHARED_COLS, S>;
                else if (nw == 16) join = MT == 1 ? forward_join_tail_kernel<T, ND, 1, 16, S> : forward_join_tail_kernel<T, ND, 2, 16, S>;
                else join = MT == 1 ? forward_join_tail_kernel<T, ND, 1, WAVESH, S> : MT == 2 ? forward_join_tail_kernel<T, ND, 2, WAVESH, S>
                          : MT == 4 || MX ? forward_join_tail_kernel<T, ND, 4, WAVESH, S> : forward_join_tail_kernel<T, ND, MX ? 4 : 8, WAVESH, S>;
                hipLaunchKernelGGL(join, dim3((unsigned)((units - whole) * (MT * TN / JOIN_ROWS))), dim3(nw * TN), 0, s, Ph, alts, sel, (const T*)part, bias, out, tsplit, (unsigned)whole, ts);
                return check_launch("forward_join_tail_kernel");
            }
            if constexpr (!S16) {
                const size_t total = (size_t)P.N * P.C_out * P.outV;
                const unsigned jb = (unsigned)((total + 255) / 256 > 4096 ? 4096 : (total + 255) / 256);
                hipLaunchKernelGGL(forward_join_partials_kernel<T>, dim3(jb), dim3(256), 0, s, part, bias, out, fsplit, total, P.C_out, P.outV);
                return check_launch("forward_join_partials_kernel");
            }
        }
    }
    if constexpr (S16) {
        if (declined) *declined = true;
        return DCN_OK;
    } else {
    T* wt = static_cast<T*>(ws);
    if (!off || transposed) {         // (the caller has another way)
        if (!declined) return fail(DCN_E_ARGUMENT, "null tensor pointer");
        *declined = true;
        return DCN_OK;
    }
    if (int rc = relayout<T>(P, w, wt, 0, s)) return rc;
    // geometry whose halo does not fit in LDS: gather straight from global memory
    P.tiles = (P.outV + WAVES * TN - 1) / (WAVES * TN);
    if ((long long)P.N * P.tiles > 0x7fffffffLL || (long long)P.G * P.mchunks > 65535)
        return fail(DCN_E_ARGUMENT, "layer too large for the kernel without LDS tiling (groups x output-channel chunks > 65535)");
    const dim3 grid((unsigned)P.N * P.tiles, (unsigned)P.G * P.mchunks);
    switch (MT) {
        case 1: hipLaunchKernelGGL((forward_kernel<T, ND, 1>), grid, dim3(WG), 0, s, P, in, off, wt, bias, out); break;
        case 2: hipLaunchKernelGGL((forward_kernel<T, ND, 2>), grid, dim3(WG), 0, s, P, in, off, wt, bias, out); break;
        case 4: hipLaunchKernelGGL((forward_kernel<T, ND, 4>), grid, dim3(WG), 0, s, P, in, off, wt, bias, out); break;
        default: hipLaunchKernelGGL((forward_kernel<T, ND, 8>), grid, dim3(WG), 0, s, P, in, off, wt, bias, out); break;
    }
    return check_launch("forward_kernel");
    }
}
}  // namespace dcn
