// CPU check of what the wavefront gather is launched with (plan_wave_gather):
// the LDS of its workgroup, for every order, rule and precision that takes it.
// Input: the binary mesh file of plan_check.cpp.  Prints per configuration
// "P<order> points <n> bytes <entry>: <words> words" or "... refused".
#include <cstdio>
#include <vector>

#include "../../polyfem_amd/csrc/plans.hpp"

using namespace pfgpu;

constexpr int CU_LDS = 163840;

// the kernel's static table and a stage per wavefront
int workgroup_lds(int order, int n_quad, int value_size, int words)
{
    const int n_local = order == 1 ? 4 : 10;
    return n_local * n_quad * 4 * value_size + wave_group(order, value_size) * words * value_size;
}

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
    int fails = 0;
    for (int n_quad : {1, 4})
        for (int vs : {8, 4}) {
            // a chunk within the cap, and the gradient's staging, fit whatever the mesh
            if (workgroup_lds(order, n_quad, vs, wave_words(order, vs)) > CU_LDS || wave_words(order, vs) > wave_limit(order, n_quad, vs) ||
                wave_rounds(order, n_quad) * 1536 / vs > wave_limit(order, n_quad, vs)) {
                std::printf("FAIL: the cap exceeds the limit\n");
                ++fails;
            }
            WavePlanHost w;
            if (!plan_wave_gather(pat, order, n_quad, en.data(), vs, w)) {
                std::printf("P%d points %d bytes %d: refused\n", order, n_quad, vs);
                continue;
            }
            std::printf("P%d points %d bytes %d: %d words\n", order, n_quad, vs, w.max_words);
            if (workgroup_lds(order, n_quad, vs, w.max_words) > CU_LDS) {
                std::printf("FAIL: %d bytes of LDS\n", workgroup_lds(order, n_quad, vs, w.max_words));
                ++fails;
            }
            // stage positions are 16-bit byte offsets; the stages are 16-byte aligned
            if (w.max_words * vs > 65536 || w.max_words % 4 != 0 || w.max_words * vs < wave_rounds(order, n_quad) * 1536) {
                std::printf("FAIL: a stage of %d words\n", w.max_words);
                ++fails;
            }
        }
    std::printf("%s\n", fails ? "FAIL" : "OK");
    return fails ? 1 : 0;
}
