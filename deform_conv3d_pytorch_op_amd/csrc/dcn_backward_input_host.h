// Host side of the backward pass to input and offset: plans and launches.
#pragma once
#include "dcn_host.h"

namespace dcn {

// The instantiations of backward_fused_kernel: channels per chunk and position tiles per block.
template <int ND, typename S>
using FusedKern = void (*)(Params, PlanSet, const unsigned*, const S*, const S*, const typename Parts<S>::Vec*, const S*, const S*, const typename Parts<S>::Vec*,
                           const float*, float*, float*, int, unsigned, int, int);
template <int ND, typename S> inline FusedKern<ND, S> fused_kernel(int cch, int tiles) {
    if (tiles == 4) return cch == 8 ? backward_fused_kernel<ND, 8, 4, S> : cch == 4 ? backward_fused_kernel<ND, 4, 4, S> : nullptr;
    if constexpr (ND == 2)
        if (cch == 16) return backward_fused_kernel<2, 16, 8, S>;
    return cch == 8 ? backward_fused_kernel<ND, 8, 8, S> : cch == 4 ? backward_fused_kernel<ND, 4, 8, S> : nullptr;
}

// The first element of grad_offset that belongs to an item from `whole` on: items are (deformable group, sample, block), blocks fastest, the
// tensor is [sample][deformable group].
template <int ND> inline size_t first_split_offset(const Params& P, long long whole) {
    const long long per_group = (long long)P.N * P.tiles, dg = whole / per_group, n = whole % per_group / P.tiles;
    if (dg >= P.DG) return (size_t)P.N * P.DG * P.kV * ND * P.outV;
    return (size_t)(dg == P.DG - 1 ? n * P.DG + dg : dg) * P.kV * ND * P.outV;
}

// S = T: the float32 / float64 operator.  S = Bf16 / Fp16 (T = float): input, weight, offset and
// grad_output are in that storage format (the gradients are float), and only the fused kernels serve
// them; where they cannot, *declined is set and nothing is launched: the caller then widens the tensors and
// runs the float32 operator.
template <typename T, int ND, typename S>
int backward_input_offset(const Geometry& g, const S* in, const S* w, const S* off, const S* gout, T* gin,
                          T* goff, void* ws, size_t ws_bytes, hipStream_t s, unsigned flags, bool* declined, Prep* given) {
    constexpr bool S16 = !std::is_same<S, T>::value;
    Params P;
    if (int rc = validate(g, P)) return rc;
    if (flags & ~(unsigned)(DCN_FLAG_OOB_OFFSET_GRAD_ZERO | FLAG_INPUT_ONLY)) return fail(DCN_E_ARGUMENT, "unknown flag");
    if (int rc = device_info(nullptr)) return rc;
    P.oob_zero = (flags & DCN_FLAG_OOB_OFFSET_GRAD_ZERO) ? 1 : 0;
    // grad_input alone (the plain convolution's backward-to-input, which is not given the input): the
    // scatter kernels need no input values; `goff` is then scratch for the one kernel that writes it anyway
    const bool input_only = (flags & FLAG_INPUT_ONLY) != 0;
    if ((!in && !input_only) || !w || !off || !gout || !gin || !goff) return fail(DCN_E_ARGUMENT, "null tensor pointer");
    bwd_data_weight_pad<T>(P.M, P.Cg, P.Mp, P.Cgp);
    DataLayout at = {};
    if (int rc = data_layout<T, S>(P, ws ? ws_bytes : 0, at)) return rc;
    const size_t wbytes = at.wbytes, tbytes = at.tbytes;
    const bool tail_words = at.tail_words;
    S* wt = static_cast<S*>(ws);
    T* in_cl = reinterpret_cast<T*>(static_cast<char*>(ws) + wbytes);
    T* gin_cl = reinterpret_cast<T*>(static_cast<char*>(ws) + wbytes + tbytes);
    const int TN = Mma<T>::TN;
    const int mk = bwd_data_mk<T>(P.M);
    float* bounds = reinterpret_cast<float*>(static_cast<char*>(ws) + at.tail_at);
    Prep own;
    Prep& prep = given ? *given : own;
    const dim3 tgrid((P.inV + 31) / 32, (unsigned)(P.C_in + 31) / 32, (unsigned)P.N), tblock(32, 8);

    // 1) one kernel: scatter privatised in LDS + coordinate gradient from an LDS input halo.
    // float32 layers whose LDS cells may be paired and 16-bit storage, of more than one tap: backward_fused_kernel, with
    // grad_output in operand order behind the channels-last regions of the workspace.  Others: backward_input_halo_kernel.
    // A halo of up to FUSED_HS cells gets the variant with that compile-time plane stride (the four
    // planes of either kind then lie within the 64 KB reach of an LDS instruction's offset field).
    // Eight wavefronts per workgroup; four (half the positions, in the block shape with the smallest
    // halo) where only that fits, e.g. under stride 2.
    constexpr int FUSED_HS = sizeof(T) == 4 ? 2720 : 2112;
    using Kern = void (*)(Params, PlanSet, const unsigned*, const S*, const S*, const S*, const S*, const float*, T*, T*, int, unsigned, int);
    struct FusedPlan {
        Params Ph;
        Kern kern;                  // null: backward_fused_kernel
        const void* entry;
        int nw, cch, csplit, goff_atomic;
        bool zero_goff, wide;
        long long whole, items, slots;
        size_t lds;
        const S* wt;
    };
    const int seg = P.cpg < P.Cg ? P.cpg : P.Cg;
    // Plans the fused kernel for a halo of margin m; false when none of its shapes fits.
    // (attempts: eight wavefronts on the default block, eight on the block shape with the smallest
    // halo, four on the block shape with the smallest halo)
    auto plan_fused = [&](int m, FusedPlan& fp) {
        for (int attempt = fused_first_waves() == 8 ? 0 : 2; attempt < 3; ++attempt) {
            int nw = attempt < 2 ? 8 : 4;
            const bool smallest = attempt > 0;
            Params Ph = P;
            // float32: two channels per LDS cell as 32-bit fixed point while the terms one cell can receive
            // (positions of the block x taps) leave at least 17 bits below the largest possible term
            const bool pair = sizeof(T) == 4 && fused_pair() && (long long)nw * TN * P.kV <= (1 << 14);
            // a single tap: a chunk is all staging and flush, which the smaller workgroups of backward_input_halo_kernel overlap
            // better, and grad_output is used once per chunk (24 layers of one tap: backward_fused_kernel takes 1.09 times as long).
            // Not where that kernel declines the output channels of a 16-bit layer.
            const bool split = pair && at.fused && (P.kV > 1 || (S16 && P.M > 256));
            int cch = 0;
            size_t lds = 0;
            Kern kern = nullptr;
            const void* entry = nullptr;
            // tiles of (tap, channel) rows that c channels take
            auto passes = [&](int c) { const int tp = Mma<T>::TN / c; return (P.kV + tp - 1) / tp; };
            if constexpr (sizeof(T) == 4) {
                // Channels per chunk and position tiles per block, the first shape that fits: more channels are fewer passes over
                // offsets, grad_offset and grad_output, and fewer tap slots (the 9 taps of a 3x3 kernel are 2 tiles per 4 channels, 3
                // per 8 or 5 per 16, the 27 of a 3x3x3 kernel 4 per 4 or 7 per 8); they are worth half as many positions to a halo
                // (128 -> 128 channels, 3x3x3, stride 1 2 2: 2.60 ms with 8 channels and 128 positions, 2.80 with 4 and 256).
                const int shapes[5][2] = {{8, 16}, {8, 8}, {4, 8}, {8, 4}, {4, 4}};
                for (int k = 0; split && attempt != 1 && k < 5 && !cch; ++k) {
                    const int tiles = shapes[k][0], cand = shapes[k][1];
                    if (tiles > nw) continue;
                    if (cand >= 8 && !(fused_chunk8() && seg >= 8 && passes(8) * 4 < passes(4) * 8)) continue;
                    if (cand == 16 && !(ND == 2 && fused_chunk16() && seg >= 16 && passes(16) * 8 < passes(8) * 16)) continue;
                    const size_t vb = fused_voxel_bytes<S>(cand), budget = fused_budget();
                    // The usual block, or the one with the smallest halo where that is a tenth smaller: zeroing, staging and flushing grow with
                    // it.  Backward passes of 60 layers of several taps, the other line's time over this one's: never the smallest halo 1.008 on
                    // average (34 -> 9, stride 1 2 2, 49 x 54 x 31 positions in binary16 1031 us : 636; 35 -> 94, stride 1 2 2, 603 : 634), where it is
                    // a fifth smaller 1.001, wherever it is smaller 0.999 (0.78 on one, 32 -> 32, two samples of 19 x 20 x 32, 270 : 346, whose
                    // blocks then fit its extents; 1.02 to 1.03 on three).
                    Params Pc = P, Ps = P;
                    const bool usual = !smallest && plan_halo<T, ND>(Pc, budget, m, cand, 1, tiles, false, 1, nullptr, 1, false);
                    if (plan_halo<T, ND>(Ps, budget, m, cand, 1, tiles, true, 1, nullptr, 1, false) && (!usual || Ps.hvol * 10 < Pc.hvol * 9)) Pc = Ps;
                    else if (!usual) continue;
                    if ((size_t)Pc.hvol * vb > budget || (long long)Pc.N * Pc.tiles * Pc.DG * 4 > 0x7fffffffLL) continue;
                    Ph = Pc;
                    cch = cand;
                    nw = tiles;
                    lds = (size_t)Ph.hstride * vb;
                    entry = reinterpret_cast<const void*>(fused_kernel<ND, S>(cand, tiles));
                }
            }
            if (split && !cch) continue;
            bool wide = false;
            if (!split) {
            const size_t chb = (pair ? 4 : 8) + sizeof(T);      // LDS bytes per channel and halo voxel: cell + input value
            // Channels per chunk: 8 where that takes fewer MFMA passes per channel (a pass holds TN / CCH
            // taps: the 9 taps of a 3x3 kernel are 2 float passes per 4 channels or 3 per 8; the 27 of a
            // 3x3x3 kernel 4 or 7) and the planes of 8 channels fit: the small halos of 2-D layers, and
            // 3-D ones with paired cells.  16 (2-D, float, paired cells): two taps per pass -- the 9 taps of
            // a 3x3 kernel are 5 passes per 16 channels instead of 6.  The float kernel with 8 channels
            // per chunk keeps the input values bank-swizzled and wants the innermost halo extent a
            // multiple of the four-channel groups per voxel.
            size_t tables = 0;
            bool fixed = false;
            for (int cand = 16; cand >= 4 && !cch; cand /= 2) {
                if (cand >= 8 && !((ND == 2 || pair) && nw == 8 && fused_chunk8() && seg >= 8 && passes(8) * 4 < passes(4) * 8)) continue;
                if (cand == 16 && !(ND == 2 && pair && fused_chunk16() && seg >= 16 && passes(16) * 8 < passes(8) * 16)) continue;
                Params Pc = P;
                const int wmult = cand == 16 ? 1 : cand == 8 ? swizzle_groups<T, 8>() : 1;
                if (!plan_halo<T, ND>(Pc, scatter_budget(), m, 8, chb, nw, smallest, 0, nullptr, wmult)) continue;
                const size_t tb = (size_t)Pc.hvol * 4;      // halo table
                if ((long long)Pc.N * Pc.tiles * Pc.DG * 4 > 0x7fffffffLL) continue;
                if (cand >= 8) {
                    if ((scatter_budget() - tb) / ((size_t)Pc.hstride * chb) < (size_t)cand) continue;
                } else {
                    // A halo of up to FUSED_HS cells gets the variant with that compile-time plane stride
                    fixed = fused_fixed_stride() && Pc.hvol <= FUSED_HS && (size_t)4 * FUSED_HS * chb + tb <= scatter_budget();
                    if (!fixed && (scatter_budget() - tb) / ((size_t)Pc.hstride * chb) < 4) continue;
                }
                Ph = Pc;
                tables = tb;
                cch = cand;
            }
            if (!cch) continue;
            const bool sixteen = cch == 16, eight = cch >= 8;
            if (fixed && !eight) Ph.hstride = FUSED_HS;
            // grad_output operand held in registers when its reduction steps fit: 32 per pass
            // (M <= 64 float, 128 double with 4-channel chunks)
            // (16-bit storage: a reduction step takes 8 output channels and an operand batch half as many steps)
            const int KS = GcolGemm<T, S>::KS, halve = S16 ? 2 : 1;
            const int ksteps = (P.M + KS - 1) / KS;
            wide = eight && !sixteen && pair && ksteps <= 32 / halve;                     // the kernel's WIDE
            const int slot_regs = (wide || sixteen) ? 8 : (Mma<T>::row(1, 0) - Mma<T>::row(0, 0) == 1) ? 4 : cch / 4;      // the kernel's RPS
            const bool breg = ksteps <= Mma<T>::NACC / slot_regs * ((wide || sixteen) ? 16 : 8) / halve;
            // float, 4-channel chunks: a second set of 32 registers takes the operand of up to 128 output channels (16-bit: 256)
            const bool breg2 = sizeof(T) == 4 && !eight && !breg && ksteps <= 64 / halve && fused_breg2();
            lds = (size_t)cch * Ph.hstride * chb + tables;
#define DCN_FUSED_C(CCH_, BREG_, HS_, NW_, PAIR_) backward_input_halo_kernel<T, ND, CCH_, true, (BREG_) || S16, HS_, NW_, true, PAIR_, 1, S>
#define DCN_FUSED_B2(HS_, NW_, PAIR_) backward_input_halo_kernel<T, ND, 4, true, true, HS_, NW_, true, PAIR_, 2, S>
            auto pick = [&](auto pair_tag) {
                constexpr bool PR = decltype(pair_tag)::value;
                if (sixteen) {
                    if constexpr (ND == 2 && PR && sizeof(T) == 4) kern = breg ? DCN_FUSED_C(16, true, 0, 8, PR) : DCN_FUSED_C(16, false, 0, 8, PR);
                } else if (eight) {
                    if constexpr (ND == 2 || PR) kern = breg ? DCN_FUSED_C(8, true, 0, 8, PR) : DCN_FUSED_C(8, false, 0, 8, PR);
                } else if (breg2) {
                    if constexpr (sizeof(T) == 4) {
                        if (nw == 8) kern = fixed ? DCN_FUSED_B2(FUSED_HS, 8, PR) : DCN_FUSED_B2(0, 8, PR);
                        else kern = fixed ? DCN_FUSED_B2(FUSED_HS, 4, PR) : DCN_FUSED_B2(0, 4, PR);
                    }
                } else if (nw == 8)
                    kern = fixed && breg ? DCN_FUSED_C(4, true, FUSED_HS, 8, PR) : fixed ? DCN_FUSED_C(4, false, FUSED_HS, 8, PR) : DCN_FUSED_C(4, false, 0, 8, PR);
                else
                    kern = fixed && breg ? DCN_FUSED_C(4, true, FUSED_HS, 4, PR) : fixed ? DCN_FUSED_C(4, false, FUSED_HS, 4, PR) : DCN_FUSED_C(4, false, 0, 4, PR);
            };
            if constexpr (sizeof(T) == 4) {
                if (pair) pick(std::true_type{});
                else pick(std::false_type{});
            } else
                pick(std::false_type{});
#undef DCN_FUSED_B2
#undef DCN_FUSED_C
            if (!kern) continue;
            if (S16 && !breg && !breg2) continue;       // 16-bit operands come from registers only
            entry = reinterpret_cast<const void*>(kern);
            }
            Ph.cchunk = cch;
            const int threads = kern ? nw * 64 : FUSED_WAVES * 64;
            // Work items are (tile, deformable group) pairs, each a run of nchunks channel chunks.  `slots`
            // workgroups run at once, so the items take whole rounds plus a partly filled last one.  Either
            // every item is split over 1, 2 or 4 workgroups (workgroup cz takes every csplit-th chunk), or
            // the items of the whole rounds stay unsplit and only those of the last round are split, as
            // finely as fills the device; they come last in the launch.  A workgroup's fixed part
            // (norms of grad_output, offsets, first loads; grad_output operand and halo table in the kernel with single cells) counts as a quarter of
            // a chunk (60 layers of several taps: a tenth, a half and a whole one within 0.1 % on average and 2 % on any; none 1.02, at worst 1.41).  The workgroups that share an item add their grad_offset parts with
            // float atomics on a zero-filled buffer; the only owner of an item stores running sums.
            const int nchunks = (seg + cch - 1) / cch;
            const long long items = (long long)Ph.N * Ph.tiles * Ph.DG;
            const long long slots = forced_slots() ? forced_slots() : resident_workgroups(entry, threads, lds);
            auto item_cost = [&](double chunks_per_wg, int wgs) { return wgs * (chunks_per_wg + 0.25) / nchunks; };
            int csplit = 1;
            long long whole = 0;                              // unsplit items at the start of the launch
            double best = 1e30;
            for (int cs = 1; cs <= 4 && cs <= nchunks; cs *= 2) {
                const double rounds = (double)((items * cs + slots - 1) / slots) / cs * item_cost((double)nchunks / cs, cs);
                if (rounds < best) { best = rounds; csplit = cs; }
            }
            if (fused_tail_split() && items > slots && items % slots) {
                const long long rest = items % slots;
                const long long cs = slots / rest < nchunks ? slots / rest : nchunks;
                if (cs >= 2) {
                    const double rounds = (double)(items / slots) * item_cost(nchunks, 1) + item_cost((double)((nchunks + cs - 1) / cs), 1);
                    if (rounds < best) { best = rounds; csplit = (int)cs; whole = items - rest; }
                }
            }
            if (forced_csplit()) { csplit = forced_csplit(); whole = 0; }
            if (csplit > nchunks) csplit = nchunks;
            if (whole + (items - whole) * csplit > 0x7fffffffLL) continue;
            fp.Ph = Ph; fp.kern = kern; fp.entry = entry; fp.nw = nw; fp.cch = cch; fp.csplit = csplit;
            // grad_offset over the chunks of an item that one workgroup owns: the running sum through plain
            // loads and stores in the 3-D kernels (float atomics run at about 3e11 per second over the device,
            // and a 3x3x3 layer has 81 grad_offset elements per position and chunk); atomics in the 2-D ones
            fp.goff_atomic = ND == 2 && nchunks > 1 ? 1 : 0;
            fp.zero_goff = fp.goff_atomic || csplit > 1;
            fp.wide = wide; fp.whole = whole; fp.items = items; fp.slots = slots; fp.lds = lds; fp.wt = nullptr;
            return true;
        }
        return false;
    };
    FusedPlan fp[MAX_PLANS];
    int margins[MAX_PLANS];
    const int nmargins = plan_margins(ND, margins);
    if (S16 && !(scatter_in_lds() && fused_coord() && !input_only && native16())) {
        if (declined) *declined = true;
        return DCN_OK;
    }
    if (scatter_in_lds() && fused_coord() && !input_only && plan_fused(margins[0], fp[0])) {
        // Wider halos for offsets that reach further; the choice is made on the device, see
        // PlanChoice.  A plan whose weights want another lane order gets a packed copy of its own in
        // the region of the channels-last input, which this path does not use.
        PlanChoice pc = {};
        pc.nplans = 1;
        pc.nd = ND;
        pc.margin[0] = margins[0];
        pc.base[0] = 1.f;
        // A sample beyond the halo scatters with global atomics.  backward_fused_kernel, 64 -> 64 channels, 4 x 16 x 56 x 56, margin 2: 1.5, 2.1, 3.1, 13,
        // 25 times the time at 25, 49, 70, 94, 98 % of the samples beyond the halo (offsets U[-r, r]; normal ones reach further: 1.2, 2.8 at 13, 45 %).
        pc.far_sample = ND == 2 ? 1.f : fp[0].kern ? 4.5f : 2.f;
        pc.far_steep = ND == 3 ? 25.f : 0.f;
        // 3-D: when most samples leave even the widest halo, the path without LDS tiling (coalesced
        // atomics on a channels-last copy; about 6.5 times the fused kernel's time on small offsets,
        // whatever the offsets) is the cheaper one: offered as a fourth choice, its kernels launched
        // behind the fused ones and gated on the choice (DCN_GLOBAL_PLAN=0: not offered)
        const bool offer_global = !S16 && ND == 3 && tail_words && global_plan() && (long long)P.N * ((P.outV + WAVES * TN - 1) / (WAVES * TN)) <= 0x7fffffffLL &&
                                  P.DG <= 65535;
        int copies = 1;                             // packed weight copies
        fp[0].wt = wt;
        for (int k = 1; k < nmargins; ++k) {
            FusedPlan& c = fp[pc.nplans];
            c.wt = nullptr;
            if (!plan_fused(margins[k], c) || c.Ph.hvol > 3 * fp[0].Ph.hvol) continue;
            for (int e = 0; e < pc.nplans && !c.wt; ++e)
                if (fp[e].cch == c.cch && fp[e].wide == c.wide && !fp[e].kern == !c.kern) c.wt = fp[e].wt;
            if (!c.wt) {
                if ((size_t)copies * wbytes > tbytes) continue;
                c.wt = reinterpret_cast<const S*>(reinterpret_cast<const char*>(in_cl) + (size_t)(copies - 1) * wbytes);
                ++copies;
            }
            pc.margin[pc.nplans] = margins[k];
            // Flush, staging and the per-chunk passes grow with the halo.  backward_fused_kernel in 3-D: with its voxels per position r, as
            // 1 + 0.008 r, a fifth more with narrower chunks (64 -> 64 channels, 4 x 16 x 56 x 56: r = 7.7, 12 and 17.7, the latter two with
            // 4-channel chunks, take 1, 1.35 and 1.36; in bfloat16 with 8-channel chunks at 12 1, 1.07 and 1.34).  With the costs above and the
            // 6.5 below, over 8 layers under 17 distributions of offsets from U[-1.5, 1.5] to U[-10, 10] the chosen plan takes 1.025 times the best one's
            // time on average; with 0.068 r, a tenth and 4.5, fitted to the loop over channels that far samples took before, 1.044.  The
            // kernel with single cells as fitted when it served them all.  Little in 2-D.
            const Params &H0 = fp[0].Ph, &Hk = c.Ph;
            const float r0 = (float)H0.hvol / (float)(fp[0].nw * TN), rk = (float)Hk.hvol / (float)(c.nw * TN);
            if (ND == 3 && !c.kern && !fp[0].kern)
                pc.base[pc.nplans] = (1.f + 0.008f * rk) / (1.f + 0.008f * r0) * (c.cch < fp[0].cch ? 1.2f : 1.f);
            else
                pc.base[pc.nplans] = (1.f + (ND == 3 ? 0.9f : 0.05f) * ((float)Hk.hvol / (float)H0.hvol - 1.f)) * (c.nw < fp[0].nw ? 1.25f : 1.f);
            ++pc.nplans;
        }
        for (int k = pc.nplans; k < MAX_PLANS; ++k) {
            pc.margin[k] = pc.margin[pc.nplans - 1];
            pc.base[k] = 1e30f;
        }
        unsigned* sel = (pc.nplans > 1 || offer_global) ? reinterpret_cast<unsigned*>(bounds + 2 * BOUND_BLOCKS + 16) : nullptr;
        pc.sel = sel;
        pc.global_cost = offer_global ? 6.5f : 0.f;
        const size_t n_off = (size_t)P.N * P.DG * P.kV * ND * P.outV;
        // one launch prepares: weights in the lane order of the kernel's operand loads, one slab per channel
        // chunk, grad_output likewise, the bounds of the weights, the choice of the plan, grad_offset cleared where
        // it is added to, and the caller's jobs
        if (sel) prep.add(PREP_PLAN, 1);
        bool any_fused = false;
        for (int k = 0; k < pc.nplans; ++k) {
            bool packed = false;
            for (int e = 0; e < k; ++e) packed = packed || fp[e].wt == fp[k].wt;
            if (packed) continue;
            const size_t slabs = (size_t)(fp[k].cch == 16 ? chunk_candidates<16>(P.cpg, P.Cg, P.C_in)
                                          : fp[k].cch == 8 ? chunk_candidates<8>(P.cpg, P.Cg, P.C_in)
                                                           : chunk_candidates<4>(P.cpg, P.Cg, P.C_in));
            const size_t total = fp[k].kern ? packed_weight_elems<T, S>(P.M, P.kV, slabs, fp[k].cch)
                                            : slabs * fused_tiles(P.kV, fp[k].cch) * fused_steps(P.M) * 64;      // threads
            PrepJob& job = prep.add(fp[k].kern ? PREP_PACK : PREP_FUSED_PACK, (unsigned)((total + 255) / 256 > 8192 ? 8192 : (total + 255) / 256));
            job.variant = fp[k].wide ? 9 : fp[k].cch;
            job.dst = const_cast<S*>(fp[k].wt);
            any_fused = any_fused || !fp[k].kern;
        }
        char* gq = static_cast<char*>(ws) + at.gq_at;
        if (any_fused) {
            const size_t total = (size_t)P.N * P.G * fused_steps(P.M) * 2 * P.outV;
            PrepJob& job = prep.add(PREP_GOUT, (unsigned)((total + 255) / 256 > 16384 ? 16384 : (total + 255) / 256));
            job.src = gout;
            job.dst = gq;
        }
        prep.add(PREP_BOUNDS, BOUND_BLOCKS).dst = bounds;
        // grad_offset is cleared from the first element that is added to: where only the last round's items are split, the last samples of the last
        // deformable group.
        size_t added = n_off;
        for (int k = 0; k < pc.nplans; ++k) {
            const size_t from = !fp[k].zero_goff ? n_off : fp[k].goff_atomic ? 0 : first_split_offset<ND>(fp[k].Ph, fp[k].whole);
            if (from < added) added = from;
        }
        if (added < n_off) prep.zero(goff + added, (n_off - added) * sizeof(T));
        // Where the fused kernel collects grad_input: in octets of channels in the place of the channels-last gradient, or in the tensor itself.  In 3-D
        // the last launch of the path without LDS tiling, or the rounding of a 16-bit layer's gradients, brings them to the tensor, and a halo
        // has 8 to 18 voxels to a position.  In 2-D it has two: steps of 256 -> 256, 3x3, 8 x 56 x 56 874 us in the tensor, 883 in octets (one launch more),
        // in binary16 435 and 436.  Halos so large that float32 chunks are half octets flush a line twice: backward passes to input and offset of 132 such layers 0.93 to 1.18 times
        // as fast as in the tensor, 1.02 on average (2x2x2 at stride 2, 64 -> 64, two samples of 16 x 56 x 56, 193 us in the tensor, 203 in octets; 4x4x4 at stride 2, 64 -> 64, one
        // sample, samples within 1.5 voxels 261 and 270, within 3 483 and 412: the corners of a sample past the halo are a line in octets).
        bool octets = ND == 3 && sizeof(T) == 4 && at.fused && tail_words && P.cpg % 8 == 0 && P.Cg % 8 == 0;
        for (int k = 0; k < pc.nplans; ++k) octets = octets && !fp[k].kern;
        if (octets) prep.zero(gin_cl, (size_t)P.N * P.C_in * P.inV * sizeof(T));
        else if (given) prep.zero(gin, (size_t)P.N * P.C_in * P.inV * sizeof(T));
        float* const collect = reinterpret_cast<float*>(octets ? gin_cl : gin);
        if (trace_plans() && ND == 3) fprintf(stderr, "dcn backward_input_offset: grad_input collected in %s\n", octets ? "octets" : "the tensor");
        if (int rc = launch_prepare<T, S>(P, pc, prep, w, off, n_off, s)) return rc;
        // one launch per set of plans that differ in nothing but the halo
        unsigned launched = 0;
        for (int k = 0; k < pc.nplans; ++k) {
            if ((launched >> k) & 1u) continue;
            // (the kernel takes plan 0 as its Params argument: a launch that does not serve plan 0 gets
            // the Params of its first plan there, which its mask never selects as such)
            PlanSet alts;
            alts.mask = 0;
            size_t lds = 0;
            for (int e = 1; e < MAX_PLANS; ++e) alts.alt[e - 1] = halo_plan_of(fp[k].Ph);
            for (int e = k; e < pc.nplans; ++e) {
                const bool same = fp[e].entry == fp[k].entry && fp[e].wt == fp[k].wt && fp[e].csplit == fp[k].csplit && fp[e].whole == fp[k].whole &&
                                  fp[e].items == fp[k].items && fp[e].goff_atomic == fp[k].goff_atomic && fp[e].nw == fp[k].nw &&
                                  fp[e].slots == fp[k].slots && same_blocks(fp[e].Ph, fp[k].Ph);      // (as many workgroups per CU with the larger LDS)
                if (!same) continue;
                if (e > 0) alts.alt[e - 1] = halo_plan_of(fp[e].Ph);
                alts.mask |= 1u << e;
                if (fp[e].lds > lds) lds = fp[e].lds;
            }
            launched |= alts.mask;
            if (trace_plans()) {
                fprintf(stderr, "dcn backward_input_offset: launch for plans %#x: %d position tiles, %d channels per chunk%s, grid %lld (%lld unsplit, rest x %d), LDS %zu\n",
                        alts.mask, fp[k].nw, fp[k].cch, fp[k].kern ? " (halo kernel)" : "", fp[k].whole + (fp[k].items - fp[k].whole) * fp[k].csplit, fp[k].whole,
                        fp[k].csplit, lds);
                for (int e = 0; e < pc.nplans; ++e)
                    if ((alts.mask >> e) & 1u)
                        fprintf(stderr, "  plan %d: margin %d, halo %d x %d x %d, base cost %.3f\n", e, pc.margin[e], fp[e].Ph.hext[0], fp[e].Ph.hext[1],
                                fp[e].Ph.hext[2], pc.base[e]);
            }
            if (lds > 48 * 1024)
                if (int rc = raise_lds_limit(fp[k].entry, lds)) return rc;
            const dim3 grid((unsigned)(fp[k].whole + (fp[k].items - fp[k].whole) * fp[k].csplit));
            if (fp[k].kern) {
                hipLaunchKernelGGL(fp[k].kern, grid, dim3(fp[k].nw * 64), lds, s, fp[k].Ph, alts, (const unsigned*)sel, in, off, fp[k].wt, gout,
                                   (const float*)bounds, gin, goff, fp[k].csplit, (unsigned)fp[k].whole, fp[k].goff_atomic);
            } else {
                if constexpr (sizeof(T) == 4) {
                    typedef const typename Parts<S>::Vec* Ops;
                    hipLaunchKernelGGL((fused_kernel<ND, S>(fp[k].cch, fp[k].nw)), grid, dim3(FUSED_WAVES * 64), lds, s, fp[k].Ph, alts, (const unsigned*)sel, in, off,
                                       reinterpret_cast<Ops>(fp[k].wt), w, gout, reinterpret_cast<Ops>(gq), (const float*)bounds, collect, goff, fp[k].csplit,
                                       (unsigned)fp[k].whole, fp[k].goff_atomic, octets ? 1 : 0);
                }
            }
            if (int rc = check_launch(fp[k].kern ? "backward_input_halo_kernel" : "backward_fused_kernel")) return rc;
        }
        if constexpr (!S16) if (offer_global) {
            // the fourth choice: three launches that return at once unless *sel == MAX_PLANS.  They reuse
            // the weight region and the channels-last regions, which the fused kernels no longer read then.
            Params Pg = P;
            Pg.tiles = (P.outV + WAVES * TN - 1) / (WAVES * TN);
            const size_t total_w = (size_t)P.G * P.kV * P.Mp * P.Cgp, pad_w = (size_t)TAP_PAD * P.Mp * P.Cgp;
            const size_t nelem = (size_t)P.N * P.C_in * P.inV;
            const unsigned nb_w = (unsigned)((total_w + pad_w + 255) / 256 > 1024 ? 1024 : (total_w + pad_w + 255) / 256);
            const unsigned nb_z = (unsigned)((nelem + 1023) / 1024 > 4096 ? 4096 : (nelem + 1023) / 1024);
            const size_t ntiles = (size_t)P.N * ((P.C_in + 31) / 32) * ((P.inV + 31) / 32);
            const unsigned nb_t = (unsigned)(ntiles > 16384 ? 16384 : ntiles);
            if (trace_plans()) fprintf(stderr, "dcn backward_input_offset: path without LDS tiling offered at cost %.2f\n", pc.global_cost);
            hipLaunchKernelGGL(global_path_prepare_kernel<T>, dim3(nb_w + nb_z + nb_t), dim3(256), 0, s, Pg, w, wt, pad_w, gin_cl, in, in_cl,
                               nb_w, nb_z, (const unsigned*)sel, (unsigned)MAX_PLANS);
            if (int rc = check_launch("global_path_prepare_kernel")) return rc;
            hipLaunchKernelGGL((backward_data_kernel<T, ND, true, 0>), dim3((unsigned)Pg.N * Pg.tiles, (unsigned)P.DG), dim3(WG), 0, s, Pg,
                               (const T*)in_cl, off, (const T*)wt, gout, gin_cl, goff, (const unsigned*)sel, (unsigned)MAX_PLANS);
            if (int rc = check_launch("backward_data_kernel")) return rc;
            if (!octets) {
                hipLaunchKernelGGL(add_from_channels_last_kernel<T>, tgrid, tblock, 0, s, (const T*)gin_cl, gin, P.C_in, P.inV,
                                   (const unsigned*)sel, (unsigned)MAX_PLANS);
                if (int rc = check_launch("add_from_channels_last_kernel")) return rc;
            }
        }
        if constexpr (sizeof(T) == 4)
            if (octets) {
                if (S16 && given) {                     // (the caller rounds them)
                    given->octets = reinterpret_cast<const float*>(gin_cl);
                    return DCN_OK;
                }
                const size_t blocks = ((size_t)P.N * (P.C_in / 8) * P.inV + 255) / 256;
                auto kernel = given ? octets_to_planes_kernel<false> : octets_to_planes_kernel<true>;
                hipLaunchKernelGGL(kernel, dim3((unsigned)(blocks < 65536 ? blocks : 65536)), dim3(256), 0, s, (const float*)gin_cl, gin, P.N, P.C_in, P.inV,
                                   (const unsigned*)(offer_global ? sel : nullptr), (unsigned)MAX_PLANS);
                return check_launch("octets_to_planes_kernel");
            }
        return DCN_OK;
    }
    if constexpr (S16) {
        if (declined) *declined = true;
        return DCN_OK;
    } else {

    // 2) grad_offset from the channels-last kernel, grad_input from the LDS-privatised scatter
    {
        if (given) prep.zero(gin, (size_t)P.N * P.C_in * P.inV * sizeof(T));
        prep.add(PREP_BOUNDS, BOUND_BLOCKS).dst = bounds;
        PlanChoice none = {};
        if (int rc = launch_prepare<T, S>(P, none, prep, w, off, 0, s)) return rc;
    }
    if (int rc = relayout<T>(P, w, wt, 1, s)) return rc;
    {   // zero tap slabs behind the last group
        const size_t used = (size_t)P.G * P.kV * P.Mp * P.Cgp, pad = (size_t)TAP_PAD * P.Mp * P.Cgp;
        hipLaunchKernelGGL(fill_zero_kernel<T>, dim3((unsigned)((pad + 255) / 256)), dim3(256), 0, s, wt + used, pad);
        if (int rc = check_launch("fill_zero_kernel")) return rc;
    }
    if (!input_only) {
        hipLaunchKernelGGL(to_channels_last_kernel<T>, tgrid, tblock, 0, s, in, in_cl, P.C_in, P.inV);
        if (int rc = check_launch("to_channels_last_kernel")) return rc;
    }
    Params Ph = P;
    bool halo = scatter_in_lds() && plan_halo<T, ND>(Ph, scatter_budget(), default_margin(), 8, 8);
    if (halo && (long long)Ph.N * Ph.tiles * Ph.DG > 0x7fffffffLL) halo = false;
    if (halo) {                                     // the scatter kernel packs 4 or 8 channels per MFMA tile
        const size_t fit = (scatter_budget() - (size_t)Ph.hvol * 4) / ((size_t)Ph.hstride * 8);
        if (fit >= 8) Ph.cchunk = 8;
        else if (fit >= 4) Ph.cchunk = 4;
        else halo = false;
    }
    P.tiles = (P.outV + WAVES * TN - 1) / (WAVES * TN);
    if ((long long)P.N * P.tiles > 0x7fffffffLL || P.DG > 65535)
        return fail(DCN_E_ARGUMENT, "layer too large for the kernel without the fused LDS halo (more than 65535 deformable groups)");
    const dim3 grid((unsigned)P.N * P.tiles, (unsigned)P.DG);
    if (halo) {
        T* none = nullptr;
        if (!input_only)
        switch (mk) {      // register-resident grad_output slab when M is small enough
            case 8: hipLaunchKernelGGL((backward_data_kernel<T, ND, false, 8>), grid, dim3(WG), 0, s, P, in_cl, off, wt, gout, none, goff); break;
            case 16: hipLaunchKernelGGL((backward_data_kernel<T, ND, false, 16>), grid, dim3(WG), 0, s, P, in_cl, off, wt, gout, none, goff); break;
            case 32: hipLaunchKernelGGL((backward_data_kernel<T, ND, false, 32>), grid, dim3(WG), 0, s, P, in_cl, off, wt, gout, none, goff); break;
            default: hipLaunchKernelGGL((backward_data_kernel<T, ND, false, 0>), grid, dim3(WG), 0, s, P, in_cl, off, wt, gout, none, goff); break;
        }
        if (!input_only)
            if (int rc = check_launch("backward_data_kernel")) return rc;
        const size_t lds = (size_t)Ph.cchunk * Ph.hstride * 8 + (size_t)Ph.hvol * 4;
        const dim3 hgrid((unsigned)Ph.N * Ph.tiles * Ph.DG);
        T* nogoff = nullptr;
        PlanSet alts;
        for (int e = 1; e < MAX_PLANS; ++e) alts.alt[e - 1] = halo_plan_of(Ph);
        alts.mask = 1u;
        const unsigned* nosel = nullptr;
        if (Ph.cchunk == 8)
            return launch_halo(backward_input_halo_kernel<T, ND, 8, false, false, 0, WAVESH>, "backward_input_halo_kernel", hgrid, WGH, lds, s,
                               Ph, alts, nosel, in, off, (const T*)wt, gout, (const float*)bounds, gin, nogoff, 1, 0u, 0);
        if (Ph.cchunk == 4)
            return launch_halo(backward_input_halo_kernel<T, ND, 4, false, false, 0, WAVESH>, "backward_input_halo_kernel", hgrid, WGH, lds, s,
                               Ph, alts, nosel, in, off, (const T*)wt, gout, (const float*)bounds, gin, nogoff, 1, 0u, 0);
        return fail(DCN_E_LAUNCH, "no scatter kernel for this channel chunk");
    }
    // halo does not fit in LDS: scatter with global atomics on the channels-last copy
    const size_t nelem = (size_t)P.N * P.C_in * P.inV;
    const unsigned fblocks = (unsigned)((nelem + 1023) / 1024 > 8192 ? 8192 : (nelem + 1023) / 1024);
    hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(fblocks), dim3(256), 0, s, gin_cl, nelem);
    if (int rc = check_launch("fill_zero_kernel")) return rc;
    if (input_only) {       // the kernel reads input values for the grad_offset it also writes (into scratch here)
        hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(fblocks), dim3(256), 0, s, in_cl, nelem);
        if (int rc = check_launch("fill_zero_kernel")) return rc;
    }
    hipLaunchKernelGGL((backward_data_kernel<T, ND, true, 0>), grid, dim3(WG), 0, s, P, in_cl, off, wt, gout, gin_cl, goff);
    if (int rc = check_launch("backward_data_kernel")) return rc;
    hipLaunchKernelGGL(add_from_channels_last_kernel<T>, tgrid, tblock, 0, s, gin_cl, gin, P.C_in, P.inV);
    return check_launch("add_from_channels_last_kernel");
    }
}


}  // namespace dcn
