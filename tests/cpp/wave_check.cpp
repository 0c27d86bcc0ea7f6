// CPU check of the wavefront gather's plan (make_wave_plan), meant to run
// under AddressSanitizer / UndefinedBehaviorSanitizer: walks every chunk as
// k_gather_wave does and checks each stage position, descriptor and output.
// Input: the binary mesh file of plan_check.cpp.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../polyfem_amd/csrc/plans.hpp"

using namespace pfgpu;

static long n_fail = 0;
#define CHECK(c, ...)                                                                                          \
    do {                                                                                                       \
        if (!(c)) {                                                                                            \
            if (n_fail++ < 20) {                                                                               \
                std::fprintf(stderr, "CHECK failed line %d: ", __LINE__);                                      \
                std::fprintf(stderr, __VA_ARGS__);                                                             \
                std::fprintf(stderr, "\n");                                                                    \
            }                                                                                                  \
        }                                                                                                      \
    } while (0)

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
    const auto &np = pat.node_ptr, &ni = pat.node_inc, &bp = pat.brow_ptr, &bc = pat.bcol;
    // the rounds the library uses: P1 two (one point) or one, P2 one
    for (int cfg = 0; cfg < 2; ++cfg) {
        const int vs = cfg == 0 ? 8 : 4; // bytes of an entry
        const int rounds = order == 1 ? 2 - cfg : 1;
        WavePlanHost w;
        if (!make_wave_plan(pat, NB, en.data(), rounds, 2528, vs, w)) {
            std::printf("rounds %d: refused\n", rounds);
            continue;
        }
        const int nc = int(w.head.size());
        std::vector<int> covered(static_cast<size_t>(N), 0);
        for (const WaveHead &h : w.head)
            for (int i = 0; i < h.n_rows; ++i) covered[size_t(h.row0 + i)]++;
        for (int i : w.unused) {
            CHECK(np[size_t(i) + 1] == np[size_t(i)], "node %d has elements but no chunk", i);
            covered[size_t(i)]++;
        }
        for (int v : covered) CHECK(v == 1, "a row lies in %d chunks", v);
        CHECK(w.dst.size() == size_t(nc) * 64 * rounds * NB, "dst size");
        for (int c = 0; c < nc; ++c) {
            const WaveHead &h = w.head[size_t(c)];
            const int nr = h.n_rows, nu = h.n_units, nb = h.n_blocks, n_short = nb - h.n_long;
            CHECK(nb >= 1 && nu == np[size_t(h.row0 + nr)] - h.unit0 && nb == bp[size_t(h.row0 + nr)] - h.blk0, "chunk %d extent", c);
            CHECK(nr >= 1 && nr <= WAVE_ROWS && nu <= 64 * rounds && nb <= WAVE_BLOCKS && h.n_long <= 64, "chunk %d: %d rows %d units %d blocks", c, nr, nu, nb);
            CHECK(h.unit0 == np[size_t(h.row0)] && h.blk0 == bp[size_t(h.row0)], "chunk %d head", c);
            CHECK(h.n_groups == (n_short + 63) / 64 && size_t(h.desc0 + 64 * h.n_groups) <= w.desc.size() &&
                      2 * size_t(h.long0 + h.n_long) <= w.long_desc.size(), "chunk %d descriptors", c);
            CHECK(w.max_words * vs <= 65536, "stage of %d words", w.max_words);
            // the stage as the lanes write it: which contribution's entry sits where
            std::vector<int> stage(size_t(w.max_words), -1); // 3 (unit * NB + b) + n
            const uint16_t *d = w.dst.data() + size_t(c) * 64 * rounds * NB;
            for (int u = 0; u < nu; ++u)
                for (int b = 0; b < NB; ++b) {
                    const int pb = d[((size_t(u / 64) * (NB / 2) + b / 2) * 64 + u % 64) * 2 + b % 2];
                    CHECK(pb % vs == 0 && pb / vs + 128 < w.max_words, "chunk %d position %d", c, pb);
                    if (pb / vs + 128 >= w.max_words) continue;
                    for (int n = 0; n < 3; ++n) {
                        int &e = stage[size_t(pb / vs + 64 * n)];
                        CHECK(e < 0, "chunk %d: position taken twice", c);
                        e = 3 * (u * NB + b) + n;
                    }
                }
            // the sums
            std::vector<int> done(size_t(nb), 0);
            auto contribution = [&](int k, int rl, int word, int &last) {
                CHECK(word >= 0 && word + 128 < w.max_words, "chunk %d block %d reads word %d", c, k, word);
                if (word < 0 || word + 128 >= w.max_words) return;
                const int at = stage[size_t(word)] / 3;
                CHECK(stage[size_t(word)] >= 0 && stage[size_t(word)] % 3 == 0 && stage[size_t(word + 64)] == 3 * at + 1 &&
                          stage[size_t(word + 128)] == 3 * at + 2, "chunk %d block %d reads an empty or foreign word", c, k);
                if (stage[size_t(word)] < 0) return;
                const int u = h.unit0 + at / NB, b = at % NB, e = ni[size_t(u)] / NB, i = h.row0 + rl;
                CHECK(en[size_t(e) * NB + ni[size_t(u)] % NB] == i && bc[size_t(h.blk0 + k)] == en[size_t(e) * NB + b],
                      "chunk %d block %d adds another block's contribution", c, k);
                CHECK(u > last, "chunk %d block %d: not in unit order", c, k);
                last = u;
            };
            const int out_words = 4 * nb;
            int base = 0, idle = 0;
            for (int t = 0; t < h.n_groups; ++t) {
                const int cm = h.count[t] & 15, least = h.count[t] >> 4;
                CHECK(t == 0 || base >= out_words, "chunk %d group %d overlaps the output area", c, t);
                CHECK(base + 192 * cm + 8 <= h.long_base, "chunk %d group %d reaches the long blocks", c, t);
                // two contributions are read at a time, the second perhaps past the group
                CHECK(base + WAVE_STEP * (cm % 2 ? cm : cm - 1) + 191 < w.max_words + 192, "chunk %d group %d reads past the stage", c, t);
                for (int l = 0; l < 64; ++l) {
                    const uint32_t v = w.desc[size_t(h.desc0 + 64 * t + l)];
                    const int k = int(v >> 4) & 1023, rl = int(v >> 14) / 4, cnt = int(v & 15u);
                    if (cnt == 0) {
                        ++idle;
                        continue;
                    }
                    CHECK(k < nb && rl < nr && cnt >= least && cnt <= cm && cnt <= WAVE_SHORT, "chunk %d descriptor", c);
                    CHECK(bp[size_t(h.row0 + rl)] <= h.blk0 + k && h.blk0 + k < bp[size_t(h.row0 + rl) + 1], "chunk %d row of block", c);
                    int last = -1;
                    for (int q = 0; q < cnt; ++q) contribution(k, rl, base + WAVE_STEP * q + l, last);
                    done[size_t(k)] += cnt;
                }
                base += 192 * cm + 8;
                if (t == 0) base = std::max(base, (out_words + 7) / 8 * 8);
            }
            CHECK(idle == 64 * h.n_groups - n_short, "chunk %d: %d idle lanes", c, idle);
            CHECK(h.long_base >= out_words && out_words <= w.max_words, "chunk %d: the long blocks overlap the output area", c);
            for (int j = 0; j < h.n_long; ++j) {
                const uint32_t v = w.long_desc[2 * size_t(h.long0 + j)], v1 = w.long_desc[2 * size_t(h.long0 + j) + 1];
                const int k = int(v >> 4) & 1023, rl = int(v >> 14) / 4, cnt = int(v1 >> 16), p0 = int(v1 & 0xffffu);
                const int pieces = (cnt + WAVE_SHORT - 1) / WAVE_SHORT;
                CHECK(k < nb && rl < nr && cnt > WAVE_SHORT && pieces <= h.max_pieces && h.max_pieces <= 21, "chunk %d long descriptor", c);
                // whole pieces are read
                CHECK(h.long_base + (p0 + pieces - 1) / 8 * 192 + 191 < w.max_words, "chunk %d long block past the stage", c);
                int last = -1;
                for (int q = 0; q < cnt; ++q) {
                    const int p = p0 + q / WAVE_SHORT;
                    contribution(k, rl, h.long_base + p / 8 * 192 + p % 8 * WAVE_SHORT + q % WAVE_SHORT, last);
                }
                done[size_t(k)] += cnt;
            }
            int total = 0;
            for (int k = 0; k < nb; ++k) {
                CHECK(done[size_t(k)] >= 1, "chunk %d block %d not summed", c, k);
                total += done[size_t(k)];
            }
            CHECK(total == nu * NB, "chunk %d: %d of %d contributions summed", c, total, nu * NB);
        }
        std::printf("rounds %d: %d chunks checked, %d stage words\n", rounds, nc, w.max_words);
    }
    std::printf("%s (%ld failures)\n", n_fail ? "FAIL" : "OK", n_fail);
    return n_fail ? 1 : 0;
}
