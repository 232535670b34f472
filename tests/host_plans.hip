// Host code of the library's planning, run on the CPU by test_host_plans.py (no GPU, nothing is launched):
//   host_plans <what> <seed> <count>     exit status 0 when the property holds for `count` random layers
#include "../deform_conv3d_pytorch_op_amd/csrc/dcn_forward_host.h"
#include "../deform_conv3d_pytorch_op_amd/csrc/dcn_backward_input_host.h"
#include "../deform_conv3d_pytorch_op_amd/csrc/dcn_backward_weight_split.h"

#include <random>

using namespace dcn;

static std::mt19937 rng;
static int pick(int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); }

static bool random_layer(int nd, Params& P) {
    Geometry g{nd, pick(1, 4), 0, 0, {1, 1, 1}, {1, 1, 1}, {1, 1, 1}, {0, 0, 0}, {1, 1, 1}, {1, 1, 1}, 0, pick(1, 3)};
    g.cpg = pick(1, 40);
    if (pick(0, 1)) g.cpg = pick(1, 4) * 4;
    g.C_in = g.cpg * pick(1, 64);
    if (g.C_in % g.G) return false;
    g.C_out = g.G * pick(1, 300);
    for (int a = 3 - nd; a < 3; ++a) {
        g.k[a] = pick(1, 5);
        g.stride[a] = pick(1, 4);
        g.dil[a] = pick(1, 4);
        g.pad[a] = pick(0, 4);
        g.in[a] = pick(4, 90);
        const int o = g.in[a] + 2 * g.pad[a] - g.k[a];
        if (o < 0) return false;
        g.out[a] = o / g.stride[a] + 1;
    }
    return validate(g, P) == DCN_OK;
}

// The allocation-free entry point's array holds the packed weights of every layer it accepts.
static bool noalloc(const Params& P, int& hits) {
    if (noalloc_weight_bytes(P) > DCN_NOALLOC_SCRATCH_BYTES) return true;
    ++hits;
    const int Mp8 = ((P.M + 31) / 32 + 7) / 8 * 8 * 32;
    return split_weight_bytes<float>(P, Mp8) + 512 <= NOALLOC_ARRAY_BYTES;
}
// 16-bit storage is served by the 16-bit kernels where a halo of float32 cells fits a block of 256 positions.
template <int ND> static bool native16(const Params& P, int& hits) {
    bool fits = false;
    for (bool smallest : {false, true}) {
        Params Pt = P;
        fits = fits || plan_halo<float, ND>(Pt, 144 * 1024, 2, 1 << 30, 4, 8, smallest, FQ, nullptr, 1, true);
    }
    hits += fits;
    return forward16_native<ND>(P) == fits;
}

// The layout of a backward_input_offset workspace: any size from the packed weights and two channels-last tensors on is taken, the
// queried size has room for the fused kernel, and no part reaches into another or past the end.
template <typename T, typename S> static bool layout_holds(const Params& P, size_t ws, bool fused) {
    DataLayout l = {};
    if (data_layout<T, S>(P, ws, l) != DCN_OK || l.fused != fused) return false;
    const size_t weights = fused ? bwd_fused_weight_bytes<T, S>(P.M, P.Cg, P.kV, P.G, P.cpg) : bwd_data_weight_bytes<T>(P.M, P.Cg, P.kV, P.G, P.cpg);
    const size_t regions = weights + 2 * align256((size_t)P.N * P.C_in * P.inV * sizeof(T)), gout = fused ? fused_gout_need<S>(P.N, P.M, P.G, P.outV) : 0;
    if (l.wbytes != weights || l.wbytes + 2 * l.tbytes != regions || regions > ws || l.tail_at + BWD_TAIL > ws || l.tail_at % 256) return false;
    return l.tail_words ? l.gq_at == regions && l.tail_at >= regions + gout : l.tail_at == l.wbytes + l.tbytes && l.tbytes >= BWD_TAIL && !fused;
}
template <typename T, typename S> static bool layout(const Params& P, int& hits) {
    const size_t tbytes = align256((size_t)P.N * P.C_in * P.inV * sizeof(T));
    const size_t least = bwd_data_weight_bytes<T>(P.M, P.Cg, P.kV, P.G, P.cpg) + 2 * tbytes + (tbytes < BWD_TAIL ? BWD_TAIL : 0);
    const size_t query = backward_data_need<T>(P.N, P.C_in, P.C_out, P.inV, P.outV, P.kV, P.G, P.cpg);
    DataLayout l = {};
    const bool more = sizeof(T) == 4 && fused_gout_need<S>(P.N, P.M, P.G, P.outV) > BWD_TAIL + 512;      // (the fused kernel takes more than the least)
    hits += more && bwd_fused_weight_bytes<T, S>(P.M, P.Cg, P.kV, P.G, P.cpg) > bwd_data_weight_bytes<T>(P.M, P.Cg, P.kV, P.G, P.cpg);
    return layout_holds<T, S>(P, query, true) && layout_holds<T, S>(P, query + 77, true) && (!more || layout_holds<T, S>(P, least, false)) &&
           data_layout<T, S>(P, bwd_data_weight_bytes<T>(P.M, P.Cg, P.kV, P.G, P.cpg) + 2 * tbytes - 1, l) == DCN_E_WORKSPACE;
}
// float64 has no rows of grad_output in operand order: the workspace of backward_weight is that of its copies, partial tiles and sums.
static bool weight64(const Params& P, int& hits) {
    const size_t tiles = (size_t)P.kV * ((P.C_in + 15) / 16), most = (4096 + tiles - 1) / tiles, splits = most < 256 ? most : 256;
    hits += P.M > 32;
    return backward_weight_need<double>(P.N, P.C_in, P.C_out, P.inV, P.outV, P.kV, P.G) ==
           align256((size_t)P.N * P.C_in * P.inV * 8) + align256((size_t)P.N * P.C_out * P.outV * 8) + align256(splits * P.kV * P.C_out * P.Cg * 8) +
               align256((size_t)P.N * last_strips(P.outV) * P.C_out * 8);
}
// What is cleared of grad_offset reaches every item that is added to, and starts with one of them where they lie in the last deformable group.
static bool added(const Params& Pin, int& hits) {
    Params P = Pin;
    P.tiles = pick(1, 5);
    const long long per_group = (long long)P.N * P.tiles, items = per_group * P.DG, whole = pick(0, (int)items);
    const size_t slab = (size_t)P.kV * 3 * P.outV, all = slab * P.N * P.DG, from = first_split_offset<3>(P, whole);
    size_t least = all;
    for (long long i = whole; i < items; ++i) {
        const size_t at = slab * (size_t)(i % per_group / P.tiles * P.DG + i / per_group);
        if (at < least) least = at;
    }
    const bool last = whole >= per_group * (P.DG - 1);
    hits += last && whole < items;
    return from <= least && (!last || from == least);
}
static bool layouts(const Params& P, int& hits) {
    int all[4] = {0, 0, 0, 0};
    const bool ok = layout<float, float>(P, all[0]) && layout<float, Bf16>(P, all[1]) && layout<float, Fp16>(P, all[2]) && layout<double, double>(P, all[3]);
    hits += all[0];
    return ok;
}

// Where the weight gradient reads 16 bytes of a corner to a lane.
static bool quads() {
    auto layer = [](int c_in, int cpg, int c_out) {
        Params P = {};
        P.N = 1; P.C_in = c_in; P.C_out = c_out; P.G = 1; P.cpg = cpg; P.DG = c_in / cpg; P.M = c_out; P.Cg = c_in;
        return P;
    };
    const Params g8 = layer(64, 8, 64), c64 = layer(64, 64, 64), odd = layer(20, 20, 64);
    return !split_quad<3, Bf16>(g8, 2, 8) && !split_quad<3, Bf16>(layer(16, 16, 48), 2, 8) && split_quad<3, Bf16>(layer(64, 8, 24), 1, 8) && split_quad<3, Fp16>(g8, 2, 8) &&
           split_quad<2, Bf16>(g8, 2, 8) && split_quad<3, Bf16>(c64, 2, 32) && split_quad<3, Bf16>(layer(32, 32, 64), 2, 16) && !split_quad<3, Bf16>(odd, 2, 16) &&
           !split_quad<3, float>(c64, 2, 32) && split_quad<2, float>(c64, 2, 32) && split_quad<2, float>(layer(256, 256, 256), 8, 32) && split_quad<2, float>(g8, 2, 8) &&
           split_quad<2, float>(odd, 2, 32) && !split_quad<2, float>(layer(42, 14, 64), 2, 16);
}
// Eight row tiles to a workgroup of the weight gradient or four: what the estimate says of layers whose times with either are known.
static bool row_tiles() {
    struct Layer { int nd, c_in, c_out, G, taps, N, positions; bool eight; };      // channels of one group, one segment each
    const Layer layers[] = {
        {3, 64, 256, 1, 27, 4, 50176, true},   {3, 64, 256, 1, 27, 2, 12544, true},  {3, 128, 256, 1, 27, 1, 6272, true},  {3, 256, 256, 1, 1, 4, 50176, true},
        {3, 135, 142, 1, 27, 1, 81700, true},  {3, 256, 256, 1, 27, 1, 1568, false}, {3, 128, 256, 1, 27, 1, 1568, false}, {3, 114, 253, 1, 27, 4, 693, false},
        {2, 256, 256, 1, 9, 8, 3136, true},    {2, 128, 256, 1, 9, 8, 3136, true},   {2, 512, 256, 2, 9, 8, 3136, true},   {2, 256, 256, 1, 9, 4, 784, false},
        {2, 128, 256, 1, 9, 2, 3136, false},   {2, 256, 256, 1, 1, 8, 3136, false},  {2, 950, 415, 2, 9, 2, 520, false},   {2, 86, 249, 1, 9, 2, 6633, false},
    };
    for (const Layer& l : layers) {
        const int items = (l.c_in + 31) / 32 * l.taps, groups = (items + 3) / 4 * l.G, tiles = (l.c_out + 31) / 32;
        const long long slabs = (long long)l.N * ((l.positions + 31) / 32);
        const size_t one = (size_t)l.taps * l.c_out * l.G * l.c_in * sizeof(float);
        const SplitCost four = split_cost((double)groups * ((tiles + 3) / 4), 768, slabs, 256, one), eight = split_cost((double)groups * ((tiles + 7) / 8), 512, slabs, 256, one);
        if (eight_tiles_pay(l.nd, four, eight) != l.eight) return printf("%d-D, %d -> %d: %g %g\n", l.nd, l.c_in, l.c_out, four.slabs + four.tiles, eight.slabs + eight.tiles), false;
    }
    return true;
}
// Rows of the plain convolution: chunks hold them all, with two row tiles to a wavefront only where that is no more padding (single taps: a quarter more).
static bool plain_row_chunks() {
    for (int M = 1; M <= 2000; ++M)
        for (int taps : {1, 9}) {
            const PlainRows r = plain_rows(M, taps);
            const int tiles = (M + 31) / 32, held = r.mw * r.rw * r.mchunks, one = tiles > 2 ? (tiles + 3) / 4 * 4 : tiles;
            if (held < tiles || (taps > 1 && held != one) || held * 4 > one * 5 || r.mw * r.rw > 8) return printf("%d rows, %d taps\n", M, taps), false;
        }
    return plain_rows(256, 9).rw == 2 && plain_rows(257, 9).rw == 1 && plain_rows(339, 1).rw == 1 && plain_rows(591, 9).rw == 1 && plain_rows(591, 1).rw == 2;
}
// Channels at a time of the plain convolution: they fit, two workgroups to a CU or one at the least channels; of one row tile, where there are many, four down to 24 channels.
static bool plain_chunks() {
    for (int i = 0; i < 20000; ++i) {
        const PlainRows r = plain_rows(pick(1, 300), 9);
        const int most = pick(1, 8) * 8, hvol = pick(1, 40) * pick(1, 40), wgs = pick(1, 4000), c = plain_channels(r, wgs, most, hvol, 256);
        const bool four = r.mw == 1 && wgs > 512;
        const size_t room = MAX_PLAIN_LDS / (four && c >= 24 && c + 8 <= most && plain_lds(hvol, c + 8) * 2 <= MAX_PLAIN_LDS ? 4 : 2);
        if (c < 8 || c > most || c % 8 || (c > 8 && plain_lds(hvol, c) > MAX_PLAIN_LDS / 2) || (four && c > 24 && plain_lds(hvol, c) > MAX_PLAIN_LDS / 4) ||
            (c < most && plain_lds(hvol, c + 8) <= room))
            return printf("%d of %d channels, %d voxels, %d workgroups\n", c, most, hvol, wgs), false;
    }
    const PlainRows one = plain_rows(15, 9), two = plain_rows(64, 9);
    return plain_channels(one, 600, 64, 144, 256) == 40 && plain_channels(one, 500, 64, 144, 256) == 64 && plain_channels(two, 600, 64, 144, 256) == 64 &&
           plain_channels(one, 600, 24, 361, 256) == 24;
}
// Which layers the kernel of the plain convolution takes: some whose times with it and with the others are known.
static bool plain_layers() {
    struct Layer { int N, h, w, c_in, c_out, k, stride, dil, G; bool faster; };
    const Layer layers[] = {
        {2, 60, 60, 256, 16, 1, 1, 1, 1, false}, {2, 60, 60, 64, 32, 3, 1, 1, 1, false}, {2, 60, 60, 64, 64, 3, 1, 1, 1, false}, {2, 60, 60, 24, 24, 5, 1, 1, 1, false},
        {2, 60, 60, 24, 24, 3, 1, 1, 1, false},  {1, 112, 112, 64, 16, 3, 1, 1, 1, false}, {16, 29, 18, 129, 56, 1, 2, 1, 1, false}, {1, 56, 56, 24, 256, 5, 1, 1, 1, false},
        {25, 24, 24, 512, 32, 3, 1, 1, 1, false}, {4, 28, 28, 128, 128, 3, 1, 1, 1, false}, {8, 24, 23, 59, 131, 3, 1, 1, 1, true}, {1, 56, 56, 64, 64, 3, 1, 1, 1, true},
        {2, 60, 60, 16, 24, 3, 1, 1, 1, true},   {2, 40, 40, 16, 128, 3, 1, 1, 1, true},  {16, 28, 28, 256, 128, 3, 1, 1, 1, true}, {8, 56, 56, 64, 64, 3, 1, 1, 1, true},
        {2, 60, 60, 8, 8, 3, 1, 1, 1, true},     {1, 82, 112, 92, 339, 3, 1, 1, 1, true},
    };
    for (const Layer& l : layers) {
        const int M = l.c_out / l.G, pad = l.k / 2 * l.dil, span = (l.k - 1) * l.dil + 1, ext = 7 * l.stride + span;
        const int oh = (l.h + 2 * pad - span) / l.stride + 1, ow = (l.w + 2 * pad - span) / l.stride + 1;
        const PlainRows r = plain_rows(M, l.k * l.k);
        if (plain_pays(r, (long long)l.N * ((oh + 7) / 8) * ((ow + 7) / 8) * l.G * r.mchunks, l.c_in / l.G, l.k * l.k, ext * ext, 256) != l.faster)
            return printf("%d -> %d, %d taps, %d of %d x %d\n", l.c_in, l.c_out, l.k * l.k, l.N, l.h, l.w), false;
    }
    return true;
}
int main(int argc, char** argv) {
    if (argc != 4) return 2;
    const std::string what = argv[1];
    rng.seed((unsigned)atoi(argv[2]));
    if (what == "jobs") {           // the list of the preparing launch takes no job too many and says so
        Prep prep;
        for (int i = 0; i < MAX_PREP; ++i) prep.add(PREP_PLAN, 1);
        const bool ok = !prep.full && prep.jobs.n == MAX_PREP && prep.blocks == (unsigned)MAX_PREP;
        prep.add(PREP_PLAN, 1);
        return ok && prep.full && prep.jobs.n == MAX_PREP ? 0 : 1;
    }
    if (what == "div") {            // what the device does with a Div is a division: up to 2^31, around multiples of every small divisor and of random ones
        auto divides = [](int d, unsigned n) {
            const Div D(d);
            return (((unsigned)((unsigned long long)D.m * n >> 32) + n) >> D.l) == n / (unsigned)d;
        };
        for (int i = 0; i < 1000 * atoi(argv[3]); ++i) {
            const int d = i < 5000 ? i + 1 : (int)(rng() % (i & 1 ? 0x7fffffffu : 100000u)) + 1;
            const unsigned n = rng() & 0x7fffffffu, m = n / d * d;
            if (!divides(d, n) || !divides(d, m) || (m && !divides(d, m - 1)) || !divides(d, 0) || !divides(d, 0x7fffffffu)) return printf("%u / %d\n", n, d), 1;
        }
        return 0;
    }
    if (what == "quad") return quads() ? 0 : 1;
    if (what == "plain_chunks") return plain_chunks() ? 0 : 1;
    if (what == "plain") return plain_layers() ? 0 : 1;
    if (what == "plain_rows") return plain_row_chunks() ? 0 : 1;
    if (what == "rows") return row_tiles() ? 0 : 1;
    if (what == "budget") {         // of any DCN_SCATTER_BUDGET_KB: what a CU has beside the 2120 and 100 bytes that the kernels declare; 72 stays 72
        const size_t cu = 160 * 1024, kb72 = 72 * 1024;
        return fused_budget() + 2120 <= cu && scatter_budget() + 100 <= cu && fused_budget() >= kb72 && scatter_budget() >= kb72 &&
                       (env_kb("DCN_SCATTER_BUDGET_KB", 0) != kb72 || (fused_budget() == kb72 && scatter_budget() == kb72))
                   ? 0 : 1;
    }
    int layers = 0, hits = 0;
    for (const int count = atoi(argv[3]); layers < count;) {
        Params P;
        const int nd = pick(2, 3);
        if (!random_layer(nd, P)) continue;
        ++layers;
        const bool ok = what == "noalloc" ? noalloc(P, hits) : what == "layout" ? layouts(P, hits) : what == "weight64" ? weight64(P, hits) : what == "added" ? added(P, hits) : what == "native16" ? (nd == 3 ? native16<3>(P, hits) : native16<2>(P, hits)) : false;
        if (!ok) {
            printf("%s: %d-D, C_in %d, C_out %d, G %d, cpg %d, k %d %d %d, stride %d %d %d, dil %d %d %d\n", what.c_str(), nd, P.C_in, P.C_out, (int)P.G, (int)P.cpg, (int)P.k[0],
                   (int)P.k[1], (int)P.k[2], P.stride[0], P.stride[1], P.stride[2], P.dil[0], P.dil[1], P.dil[2]);
            return 1;
        }
    }
    printf("%d of %d layers\n", hits, layers);
    return hits > layers / 50 && hits < layers ? 0 : 3;       // (both sides of the line were met)
}
