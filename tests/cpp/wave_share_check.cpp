// CPU check of which meshes the wavefront gather is chosen for (the rule of
// wave_plan_ready).  Input: the binary mesh file of plan_check.cpp.  Prints per
// points and bytes of an entry "points <n> bytes <entry>: share <s> chosen" or
// "... refused".
#include <cstdio>
#include <vector>

#include "../../polyfem_amd/csrc/plans.hpp"

using namespace pfgpu;

int main(int argc, char **argv)
{
    FILE *f = argc < 2 ? nullptr : std::fopen(argv[1], "rb");
    int32_t hdr[4];
    if (!f || std::fread(hdr, 4, 4, f) != 4) return 2;
    const int order = hdr[0], E = hdr[1], N = hdr[2], Nv = hdr[3], NB = order == 1 ? 4 : 10;
    std::vector<int32_t> en(size_t(E) * NB), ev(size_t(E) * 4);
    if (std::fread(en.data(), 4, en.size(), f) != en.size() || std::fread(ev.data(), 4, ev.size(), f) != ev.size()) return 2;
    std::fclose(f);
    const Pattern pat = build_pattern(E, NB, en.data(), N, Nv, ev.data());
    for (int n_quad : {1, 4})
        for (int vs : {8, 4}) {
            const double least = least_wave_share(pat, order, n_quad, vs);
            WavePlanHost w;
            const bool chosen = least <= 1 && plan_wave_gather(pat, order, n_quad, en.data(), vs, w, least);
            std::printf("points %d bytes %d: share %.3f %s\n", n_quad, vs, w.share, chosen ? "chosen" : "refused");
            // the share does not depend on the limit, and a plan's content neither
            WavePlanHost all;
            if (chosen != (least <= 1 && plan_wave_gather(pat, order, n_quad, en.data(), vs, all) && all.share >= least) ||
                (chosen && (all.dst != w.dst || all.desc != w.desc || all.share != w.share)))
                return 1;
        }
    return 0;
}
