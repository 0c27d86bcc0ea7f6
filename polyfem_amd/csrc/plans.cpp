// Host-side construction of the row-unit gather plan of the factored
// Hessian route (the kernel is k_gather_units in plain.hip).  Host code
// only, so that tests can build and check the plans on the CPU.
#include <algorithm>
#include <atomic>
#include <utility>

#include "parallel.hpp"
#include "plans.hpp"

namespace pfgpu {

namespace {

// a piece of a chunk's block sums: block (chunk-local), piece within the
// block, the block's row (chunk-local), contributions, first piece of a
// split block
struct Piece {
    int32_t block, piece, row, len;
    bool head;
};
// the cost of a piece in contributions read: its reads plus the storing of
// its sum (one block, to the values or to the stage)
constexpr int PIECE_COST = 3;

// greedy runs of consecutive pieces of at most bound cost and at most two
// heads each: the number of runs (and their first pieces)
int piece_runs(const std::vector<Piece> &p, int bound, std::vector<int> *first)
{
    int n = 0, cur = 0, heads = 0;
    for (size_t i = 0; i < p.size(); ++i) {
        const int c = p[i].len + PIECE_COST;
        if (n == 0 || cur + c > bound || (p[i].head && heads == 2)) {
            ++n;
            cur = 0;
            heads = 0;
            if (first) first->push_back(int(i));
        }
        cur += c;
        heads += p[i].head ? 1 : 0;
    }
    return n;
}

// the threads' runs of pieces in one chunk: the least maximal run cost for
// which gs threads suffice, written as gs + 1 lane entries
void chunk_lanes(const std::vector<Piece> &p, int nb, int nr, int gs, uint32_t *lanes)
{
    int lo = 0, hi = 0;
    for (const Piece &x : p) {
        lo = std::max(lo, x.len + PIECE_COST);
        hi += x.len + PIECE_COST;
    }
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (piece_runs(p, mid, nullptr) <= gs)
            hi = mid;
        else
            lo = mid + 1;
    }
    std::vector<int> first;
    piece_runs(p, lo, &first);
    for (int t = 0; t <= gs; ++t) {
        if (t < int(first.size())) {
            const Piece &x = p[size_t(first[size_t(t)])];
            lanes[t] = unit_lane(x.block, x.piece, x.row);
        } else {
            lanes[t] = unit_lane(nb, 0, nr);
        }
    }
}

} // namespace

bool make_unit_plan(const Pattern &pat, int n_local, const int32_t *elem_nodes, int gs, int n_lanes,
                    UnitPlanHost &out)
{
    const std::vector<int32_t> &np = pat.node_ptr, &ni = pat.node_inc, &bp = pat.brow_ptr, &bc = pat.bcol;
    const int NB = n_local, N = pat.n_nodes;
    // chunks of whole rows: at most gs units and gs - 1 rows each (a thread
    // per row boundary)
    std::vector<int32_t> c{0};
    int units = 0, rows = 0;
    for (int i = 0; i < N; ++i) {
        const int ui = np[size_t(i) + 1] - np[size_t(i)];
        if (ui > std::min(gs, 255)) return false;
        if (units + ui > gs || rows + 1 > gs - 1) {
            c.push_back(i);
            units = 0;
            rows = 0;
        }
        units += ui;
        rows += 1;
    }
    c.push_back(N);
    const int nc = int(c.size()) - 1;
    std::vector<uint16_t> q0(size_t(pat.n_blocks)), dst(size_t(np[size_t(N)]) * NB);
    std::vector<uint32_t> lanes(size_t(nc) * size_t(n_lanes + 1));
    std::atomic<bool> fits{true};
    // per chunk: every block's contributions are consecutive stage positions
    // (blocks in pattern order, contributions in unit order); a unit's block
    // b goes to the next free position of block (row, node_e(b))
    auto fill = [&](int c0, int c1) {
        std::vector<int32_t> cnt;
        std::vector<Piece> pieces;
        for (int ci = c0; ci < c1; ++ci) {
            int run = 0;
            for (int i = c[size_t(ci)]; i < c[size_t(ci) + 1]; ++i) {
                const int32_t r0 = bp[size_t(i)], deg = bp[size_t(i) + 1] - r0;
                const int32_t *cols = bc.data() + r0;
                auto pos = [&](int32_t j) { return int32_t(std::lower_bound(cols, cols + deg, j) - cols); };
                cnt.assign(size_t(deg), 0);
                for (int32_t u = np[size_t(i)]; u < np[size_t(i) + 1]; ++u) {
                    const int32_t e = ni[size_t(u)] / NB;
                    for (int b = 0; b < NB; ++b) cnt[size_t(pos(elem_nodes[size_t(e) * NB + b]))]++;
                }
                for (int32_t k = 0; k < deg; ++k) {
                    q0[size_t(r0 + k)] = uint16_t(run);
                    run += cnt[size_t(k)];
                    cnt[size_t(k)] = 0;
                }
                for (int32_t u = np[size_t(i)]; u < np[size_t(i) + 1]; ++u) {
                    const int32_t e = ni[size_t(u)] / NB;
                    for (int b = 0; b < NB; ++b) {
                        const int32_t k = pos(elem_nodes[size_t(e) * NB + b]);
                        dst[size_t(u) * NB + b] = uint16_t(q0[size_t(r0 + k)] + cnt[size_t(k)]++);
                    }
                }
            }
            // the pieces of the chunk's block sums, in block order
            const int i0 = c[size_t(ci)], i1 = c[size_t(ci) + 1], B0 = bp[size_t(i0)], nb = bp[size_t(i1)] - B0;
            if (nb > 4095 || i1 - i0 > 4095) {
                fits = false;
                continue;
            }
            pieces.clear();
            for (int i = i0; i < i1; ++i)
                for (int32_t blk = bp[size_t(i)]; blk < bp[size_t(i) + 1]; ++blk) {
                    const int k = blk - B0, start = q0[size_t(blk)];
                    const int n = (k + 1 < nb ? int(q0[size_t(blk) + 1]) : run) - start;
                    const int pc = n <= UNIT_PIECE ? 1 : (n + UNIT_PIECE - 1) / UNIT_PIECE;
                    for (int j = 0; j < pc; ++j)
                        pieces.push_back(Piece{k, j, i - i0, std::min(UNIT_PIECE, n - j * UNIT_PIECE), j == 0 && pc > 1});
                }
            chunk_lanes(pieces, nb, i1 - i0, n_lanes, lanes.data() + size_t(ci) * size_t(n_lanes + 1));
        }
    };
    parallel_ranges(nc, fill);
    if (!fits) return false;
    out.chunk_row = std::move(c);
    out.udst = std::move(dst);
    out.bq0 = std::move(q0);
    out.lanes = std::move(lanes);
    return true;
}

namespace {

// the stage that a chunk's contribution counts (descending) need
struct WaveShape {
    int n_long = 0, n_groups = 0, long_base = 0, max_pieces = 0, words = 0;
    uint8_t count[WAVE_GROUPS] = {};
    int base[WAVE_GROUPS] = {};
};
WaveShape wave_shape(const std::vector<int32_t> &cnt)
{
    WaveShape s;
    const int nb = int(cnt.size()), out_words = (4 * nb + 7) / 8 * 8;
    int pieces = 0;
    for (; s.n_long < nb && cnt[size_t(s.n_long)] > WAVE_SHORT; ++s.n_long) {
        const int p = (cnt[size_t(s.n_long)] + WAVE_SHORT - 1) / WAVE_SHORT;
        pieces += p;
        s.max_pieces = std::max(s.max_pieces, p);
    }
    int word = 0;
    for (int k = s.n_long; k < nb; k += 64, ++s.n_groups) {
        const int most = cnt[size_t(k)], least = cnt[size_t(std::min(k + 63, nb - 1))];
        s.base[s.n_groups] = word;
        s.count[s.n_groups] = uint8_t(most | least << 4);
        word += 192 * most + 8;
        if (s.n_groups == 0) word = std::max(word, out_words);
    }
    s.long_base = std::max(word, out_words);
    s.words = s.long_base + (pieces + 7) / 8 * 192;
    return s;
}

} // namespace

bool make_wave_plan(const Pattern &pat, int n_local, const int32_t *elem_nodes, int rounds, int word_cap,
                    int value_size, WavePlanHost &out, int word_limit, double least_share)
{
    const std::vector<int32_t> &np = pat.node_ptr, &ni = pat.node_inc, &bp = pat.brow_ptr, &bc = pat.bcol;
    const int NB = n_local, N = pat.n_nodes, cap = 64 * rounds;
    // contributions per block, and every unit's block positions in its row
    std::vector<uint8_t> count(size_t(pat.n_blocks));
    std::vector<uint16_t> upos(size_t(np[size_t(N)]) * NB);
    std::atomic<bool> fits{true};
    parallel_ranges(N, [&](int i0, int i1) {
        for (int i = i0; i < i1; ++i) {
            const int32_t r0 = bp[size_t(i)], deg = bp[size_t(i) + 1] - r0;
            if (np[size_t(i) + 1] - np[size_t(i)] > cap || deg > WAVE_BLOCKS) {
                fits = false;
                return;
            }
            const int32_t *cols = bc.data() + r0;
            for (int32_t u = np[size_t(i)]; u < np[size_t(i) + 1]; ++u) {
                const int32_t e = ni[size_t(u)] / NB;
                for (int b = 0; b < NB; ++b) {
                    const int p = int(std::lower_bound(cols, cols + deg, elem_nodes[size_t(e) * NB + b]) - cols);
                    upos[size_t(u) * NB + b] = uint16_t(p);
                    count[size_t(r0 + p)]++;
                }
            }
        }
    });
    if (!fits) return false;
    // chunks of whole rows: as many nodes as the cheap limits allow, given
    // back while the chunk's stage exceeds the cap
    std::vector<WaveHead> head;
    std::vector<int32_t> cnt;
    int64_t nw = 0, nl = 0;
    for (int i = 0; i < N;) {
        int j = i + 1;
        while (j < N && j - i < WAVE_ROWS && np[size_t(j) + 1] - np[size_t(i)] <= cap &&
               bp[size_t(j) + 1] - bp[size_t(i)] <= WAVE_BLOCKS)
            ++j;
        WaveShape s;
        int32_t hist[256] = {}; // blocks of every count
        for (int32_t b = bp[size_t(i)]; b < bp[size_t(j)]; ++b) ++hist[count[size_t(b)]];
        while (true) {
            cnt.clear();
            for (int c = cap; c >= 0; --c) cnt.insert(cnt.end(), size_t(hist[c]), c);
            s = wave_shape(cnt);
            if (j == i + 1 || (s.words <= word_cap && s.n_long <= 64)) break;
            --j;
            for (int32_t b = bp[size_t(j)]; b < bp[size_t(j) + 1]; ++b) --hist[count[size_t(b)]];
        }
        if (s.n_long > 64 || s.words > word_limit) return false;
        WaveHead h{};
        h.row0 = i;
        h.unit0 = np[size_t(i)];
        h.blk0 = bp[size_t(i)];
        h.desc0 = int32_t(nw);
        h.n_rows = j - i;
        h.n_units = np[size_t(j)] - h.unit0;
        h.n_blocks = bp[size_t(j)] - h.blk0;
        h.n_long = s.n_long;
        h.long0 = int32_t(nl);
        h.long_base = s.long_base;
        h.n_groups = s.n_groups;
        h.max_pieces = s.max_pieces;
        std::copy(s.count, s.count + WAVE_GROUPS, h.count);
        if (h.n_blocks) {
            nw += 64 * s.n_groups;
            nl += s.n_long;
            if (nw >= (int64_t(1) << 31) || s.words * value_size > 65536) return false;
            out.max_words = std::max(out.max_words, s.words);
            head.push_back(h);
        } else {
            for (int k = i; k < j; ++k) out.unused.push_back(k);
        }
        i = j;
        // the share if the rest filled its chunks; in the end, the share
        const double chunks = double(head.size()) + double(np[size_t(N)] - np[size_t(i)]) / cap;
        out.share = chunks > 0 ? double(np[size_t(N)]) / (chunks * cap) : 1.0;
        if (out.share < least_share) return false;
    }
    const int nc = int(head.size());
    std::vector<uint32_t> desc(static_cast<size_t>(nw), 0), long_desc(size_t(2 * nl));
    std::vector<uint16_t> dst(size_t(nc) * size_t(cap) * size_t(NB), 0);
    parallel_ranges(nc, [&](int c0, int c1) {
        // per output block: its contributions (unit, b), in unit order
        std::vector<int32_t> ptr, list, order, next, sorted, row_of, pos(size_t(cap) * size_t(NB));
        for (int ci = c0; ci < c1; ++ci) {
            WaveHead &h = head[size_t(ci)];
            const int nb = h.n_blocks, B0 = h.blk0;
            ptr.assign(size_t(nb) + 1, 0);
            for (int k = 0; k < nb; ++k) ptr[size_t(k) + 1] = ptr[size_t(k)] + count[size_t(B0 + k)];
            list.resize(size_t(ptr[size_t(nb)]));
            order.resize(size_t(nb));
            row_of.resize(size_t(nb));
            next.assign(ptr.begin(), ptr.end() - 1);
            for (int i = h.row0; i < h.row0 + h.n_rows; ++i) {
                for (int32_t b = bp[size_t(i)]; b < bp[size_t(i) + 1]; ++b) row_of[size_t(b - B0)] = i - h.row0;
                for (int32_t u = np[size_t(i)]; u < np[size_t(i) + 1]; ++u)
                    for (int b = 0; b < NB; ++b) {
                        const int k = bp[size_t(i)] - B0 + upos[size_t(u) * NB + b];
                        list[size_t(next[size_t(k)]++)] = (u - h.unit0) * NB + b;
                    }
            }
            // by descending count, the blocks of a count in their order
            int32_t place[257] = {};
            for (int k = 0; k < nb; ++k) ++place[count[size_t(B0 + k)]];
            for (int c = cap, at = 0; c >= 0; --c) at += std::exchange(place[c], at);
            for (int k = 0; k < nb; ++k) order[size_t(place[count[size_t(B0 + k)]]++)] = k;
            sorted.resize(size_t(nb));
            for (int j = 0; j < nb; ++j) sorted[size_t(j)] = count[size_t(B0 + order[size_t(j)])];
            const WaveShape s = wave_shape(sorted);
            auto word = [&](int k) { return uint32_t(k) << 4 | uint32_t(4 * row_of[size_t(k)]) << 14; };
            int pieces = 0;
            for (int j = 0; j < h.n_long; ++j) {
                const int k = order[size_t(j)], n = sorted[size_t(j)];
                long_desc[2 * size_t(h.long0 + j)] = word(k);
                long_desc[2 * size_t(h.long0 + j) + 1] = uint32_t(pieces) | uint32_t(n) << 16;
                for (int q = 0; q < n; ++q) {
                    const int p = pieces + q / WAVE_SHORT;
                    pos[size_t(list[size_t(ptr[size_t(k)] + q)])] = h.long_base + p / 8 * 192 + p % 8 * WAVE_SHORT + q % WAVE_SHORT;
                }
                pieces += (n + WAVE_SHORT - 1) / WAVE_SHORT;
            }
            // banks[level][instruction and half wavefront]: the banks used
            // more than `level` times; octet[group][lanes / 8]: the output
            // banks (blocks modulo 8) its eight lanes store to
            uint32_t banks[3][40] = {};
            uint8_t octet[WAVE_GROUPS][8] = {};
            auto instr = [&](int v) { return (v % NB * rounds + v / NB / 64) * 2 + v / NB % 64 / 32; };
            uint64_t free_lanes[WAVE_GROUPS];
            int least[WAVE_GROUPS];
            std::fill(free_lanes, free_lanes + WAVE_GROUPS, ~uint64_t(0));
            std::fill(least, least + WAVE_GROUPS, WAVE_SHORT);
            uint32_t *dc = desc.data() + h.desc0;
            for (int j = h.n_long; j < nb; ++j) {
                const int k = order[size_t(j)], n = sorted[size_t(j)];
                int best = 8, to = -1, lane = 0;
                for (int g = 0; g < h.n_groups && best > 0; ++g) {
                    if (n > (s.count[g] & 15) || (n < s.count[g] >> 4 && to >= 0)) continue;
                    // banks taken (once, twice, three times) by the instructions
                    // of the block's contributions, shifted back to its lane
                    uint32_t used[4] = {0, 0, 0, 0};
                    for (int q = 0; q < n; ++q) {
                        const int x = instr(list[size_t(ptr[size_t(k)] + q)]), by = (s.base[g] + q) % 32;
                        for (int lv = 0; lv < 3; ++lv) used[lv] |= by ? banks[lv][x] >> by | banks[lv][x] << (32 - by) : banks[lv][x];
                    }
                    uint64_t clash = 0;
                    for (int o = 0; o < 8; ++o)
                        if (octet[g][o] >> (k % 8) & 1) clash |= uint64_t(255) << (8 * o);
                    for (int cost = 0; cost < best; ++cost) {
                        const uint32_t u = used[cost / 2];
                        uint64_t pick = free_lanes[g] & ~(uint64_t(u) << 32 | u);
                        if (cost % 2 == 0) pick &= ~clash;
                        if (pick) {
                            best = cost;
                            to = g;
                            lane = __builtin_ctzll(pick);
                        }
                    }
                }
                free_lanes[to] &= ~(uint64_t(1) << lane);
                octet[to][lane / 8] |= uint8_t(1 << (k % 8));
                least[to] = std::min(least[to], n);
                for (int q = 0; q < n; ++q) {
                    const int v = list[size_t(ptr[size_t(k)] + q)], x = instr(v), w = s.base[to] + WAVE_STEP * q + lane;
                    const uint32_t bit = uint32_t(1) << (w % 32);
                    for (int lv = 2; lv > 0; --lv) banks[lv][x] |= banks[lv - 1][x] & bit;
                    banks[0][x] |= bit;
                    pos[size_t(v)] = w;
                }
                dc[64 * to + lane] = word(k) | uint32_t(n);
            }
            for (int g = 0; g < h.n_groups; ++g) h.count[g] = uint8_t((h.count[g] & 15) | least[g] << 4);
            uint16_t *d = dst.data() + size_t(ci) * size_t(cap) * size_t(NB);
            for (int v = 0; v < h.n_units; ++v)
                for (int b = 0; b < NB; ++b)
                    // pairs of positions share a word, words of the lanes adjacent
                    d[((size_t(v / 64) * (NB / 2) + b / 2) * 64 + v % 64) * 2 + b % 2] = uint16_t(pos[size_t(v) * NB + b] * value_size);
        }
    });
    out.head = std::move(head);
    out.dst = std::move(dst);
    out.desc = std::move(desc);
    out.long_desc = std::move(long_desc);
    return true;
}

bool plan_wave_gather(const Pattern &pat, int order, int n_quad, const int32_t *elem_nodes, int value_size, WavePlanHost &out,
                      double least_share)
{
    const int rounds = wave_rounds(order, n_quad);
    if (!make_wave_plan(pat, order == 1 ? 4 : 10, elem_nodes, rounds, wave_words(order, value_size), value_size, out,
                        wave_limit(order, n_quad, value_size), least_share))
        return false;
    out.max_words = (std::max(out.max_words, rounds * 1536 / value_size) + 3) / 4 * 4;
    return true;
}

double least_wave_share(const Pattern &pat, int order, int n_quad, int value_size)
{
    bool large = false;
    for (int i = 0; i < pat.n_nodes; ++i) large |= pat.node_ptr[size_t(i) + 1] - pat.node_ptr[size_t(i)] > 64;
    return wave_share(order, n_quad, value_size, large);
}

bool segment_chunks(const int32_t *ptr, int64_t n, int cap, std::vector<int32_t> &c)
{
    c.assign(1, 0);
    int64_t k0 = ptr[0];
    for (int64_t i = 0; i < n; ++i) {
        if (ptr[i + 1] - ptr[i] > cap) return false;
        if (ptr[i + 1] - k0 > cap) {
            c.push_back(int32_t(i));
            k0 = ptr[i];
        }
    }
    c.push_back(int32_t(n));
    return true;
}

bool make_row_plan(const Pattern &pat, RowPlanHost &out)
{
    const std::vector<int32_t> &ptr = pat.node_ptr, &inc = pat.node_inc;
    std::vector<int32_t> c;
    if (!segment_chunks(ptr.data(), pat.n_nodes, ROW_SEG, c)) return false;
    const int nc = int(c.size()) - 1;
    std::vector<int32_t> slot(size_t(nc) * ROW_SEG, -1), rmeta(size_t(pat.n_nodes));
    for (int ci = 0; ci < nc; ++ci) {
        const int32_t k0 = ptr[size_t(c[size_t(ci)])];
        for (int32_t i = c[size_t(ci)]; i < c[size_t(ci) + 1]; ++i) {
            rmeta[size_t(i)] = (ptr[size_t(i)] - k0) | ((ptr[size_t(i) + 1] - ptr[size_t(i)]) << 10);
            for (int32_t k = ptr[size_t(i)]; k < ptr[size_t(i) + 1]; ++k)
                slot[size_t(ci) * ROW_SEG + size_t(k - k0)] = inc[size_t(k)];
        }
    }
    out.chunk = std::move(c);
    out.slot = std::move(slot);
    out.rmeta = std::move(rmeta);
    return true;
}

bool make_contrib_plan(const Pattern &pat, const std::vector<int32_t> &ptr, const std::vector<int32_t> &words,
                       const std::vector<int32_t> *keys, int gs, ContribPlanHost &out)
{
    std::vector<int32_t> c;
    if (!segment_chunks(ptr.data(), pat.n_blocks, gs, c)) return false;
    const int nc = int(c.size()) - 1;
    std::vector<int32_t> slot(size_t(nc) * gs, -1), meta(size_t(pat.n_blocks));
    for (int i = 0; i < pat.n_nodes; ++i) {
        const int32_t deg = pat.brow_ptr[size_t(i) + 1] - pat.brow_ptr[size_t(i)];
        if (deg > 4095) return false;
        for (int32_t b = pat.brow_ptr[size_t(i)]; b < pat.brow_ptr[size_t(i) + 1]; ++b) meta[size_t(b)] = deg << 20;
    }
    std::vector<uint16_t> dst(keys ? size_t(nc) * gs : 0, 0);
    // chunks are independent: fill them on the host's threads
    auto fill = [&](int c0, int c1) {
        std::vector<int64_t> kv;
        std::vector<int32_t> w;
        for (int ci = c0; ci < c1; ++ci) {
            const int32_t k0 = ptr[size_t(c[size_t(ci)])], n = ptr[size_t(c[size_t(ci) + 1])] - k0;
            int32_t *sl = slot.data() + size_t(ci) * gs;
            for (int32_t b = c[size_t(ci)]; b < c[size_t(ci) + 1]; ++b) {
                meta[size_t(b)] |= (ptr[size_t(b)] - k0) | ((ptr[size_t(b) + 1] - ptr[size_t(b)]) << 10);
                for (int32_t k = ptr[size_t(b)]; k < ptr[size_t(b) + 1]; ++k) sl[k - k0] = words[size_t(k)];
            }
            if (!keys) continue;
            // the chunk's slots ordered by key (element), ties in block order,
            // with the block-order position of every contribution
            kv.resize(size_t(n));
            w.assign(sl, sl + n);
            for (int32_t i = 0; i < n; ++i) kv[size_t(i)] = (int64_t((*keys)[size_t(k0 + i)]) << 16) | i;
            std::sort(kv.begin(), kv.end());
            for (int32_t i = 0; i < n; ++i) {
                const int32_t o = int32_t(kv[size_t(i)] & 0xffff);
                sl[i] = w[size_t(o)];
                dst[size_t(ci) * gs + size_t(i)] = uint16_t(o);
            }
        }
    };
    parallel_ranges(nc, fill);
    out.chunk = std::move(c);
    out.slot = std::move(slot);
    out.meta = std::move(meta);
    out.dst = std::move(dst);
    return true;
}

} // namespace pfgpu
