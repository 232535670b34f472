// Host code of the library's planning, run on the CPU by test_host_plans.py (no GPU, nothing is launched):
//   host_plans <what> <seed> <count>     exit status 0 when the property holds for `count` random layers
#include "../deform_conv3d_pytorch_op_amd/csrc/dcn_forward_host.h"

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
    int layers = 0, hits = 0;
    for (const int count = atoi(argv[3]); layers < count;) {
        Params P;
        const int nd = pick(2, 3);
        if (!random_layer(nd, P)) continue;
        ++layers;
        const bool ok = what == "noalloc" ? noalloc(P, hits) : what == "native16" ? (nd == 3 ? native16<3>(P, hits) : native16<2>(P, hits)) : false;
        if (!ok) {
            printf("%s: %d-D, C_in %d, C_out %d, G %d, cpg %d, k %d %d %d, stride %d %d %d, dil %d %d %d\n", what.c_str(), nd, P.C_in, P.C_out, P.G, P.cpg, P.k[0],
                   P.k[1], P.k[2], P.stride[0], P.stride[1], P.stride[2], P.dil[0], P.dil[1], P.dil[2]);
            return 1;
        }
    }
    printf("%d of %d layers\n", hits, layers);
    return hits > layers / 50 && hits < layers ? 0 : 3;       // (both sides of the line were met)
}
