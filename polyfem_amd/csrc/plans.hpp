// Host-side gather plans (plans.cpp), shared by the library and the CPU
// checks of the plans.
#pragma once

#include <cstdint>
#include <vector>

#include "common.hpp"

namespace pfgpu {

// Row-unit plan of the factored gather for workgroups of gs threads: a unit
// is a node incidence (node_inc order: rows in node order, each row's
// elements in element order); chunk_row[c] .. chunk_row[c+1]-1 are the rows
// of chunk c (at most gs units and gs - 1 rows); udst[u n_local + b] is the
// stage position, within u's chunk, of u's block (row, node_e(b)); bq0[blk]
// is the first stage position of pattern block blk within its chunk (a
// block's contributions are consecutive, in unit order).
//
// The sums of a chunk's blocks are split into pieces: a block of n
// contributions is one piece when n <= UNIT_PIECE, else ceil(n / UNIT_PIECE)
// pieces of UNIT_PIECE consecutive contributions (the last shorter); a split
// block is the sum of its piece sums in piece order, each piece summed in
// unit order.  The pieces depend on n alone, so the summation order of a
// block does not depend on gs.  lanes[c (n_lanes + 1) + t] is the first
// piece of thread t of the n_lanes summing threads in chunk c (threads take
// consecutive runs of pieces, balanced by contributions; entry n_lanes is the
// end), packed by unit_lane(): the block
// (chunk-local), the piece within the block and the block's row
// (chunk-local).  A thread's run holds the first piece of at most two split
// blocks.  False when a row has more than min(gs, 255) units.
constexpr int UNIT_PIECE = 8;
constexpr uint32_t unit_lane(int block, int piece, int row)
{
    return uint32_t(block) | uint32_t(piece) << 12 | uint32_t(row) << 20;
}
struct UnitPlanHost {
    std::vector<int32_t> chunk_row;
    std::vector<uint16_t> udst, bq0;
    std::vector<uint32_t> lanes;
};
bool make_unit_plan(const Pattern &pat, int n_local, const int32_t *elem_nodes, int gs, int n_lanes,
                    UnitPlanHost &out);

// Wavefront plan of the factored gather (k_gather_wave in gather.hip): a
// chunk is a run of whole node rows with at most 64 rounds units, WAVE_ROWS
// rows and WAVE_BLOCKS pattern blocks, gathered by one wavefront.  A unit is a
// node incidence as above; unit v of the chunk is formed by lane v % 64 of
// round v / 64.
//
// The wavefront stages the three entries of a row of every contribution in
// LDS and adds them by descending count of contributions, so that its lanes
// add alike.  The short blocks (at most WAVE_SHORT contributions) are dealt
// 64 at a time to the lanes; entry n of contribution k of the block on lane l
// of group g sits at word base_g + WAVE_STEP k + 64 n + l: the lanes read
// their sums without bank conflicts and with no index arithmetic, and a group
// whose largest count is c takes 192 c + 8 words.  The lane of a block, and
// its group where several hold its count, are chosen so that the words one
// store instruction fills lie in different LDS banks as far as possible;
// WAVE_STEP = 193 instead of 192 parts the contributions that one block gets
// from one instruction (P2: 1.9 cycles per store of 32 lanes where the first
// free lane takes 3.4 and the choice without the extra word 2.8; P1: 2.0
// where it takes 3.8).  The long blocks' contributions follow from word
// long_base in pieces of WAVE_SHORT, eight pieces per 192 words.  The sums go
// to an output area of 4 words per block that overlaps group 0; group 1
// starts behind it.
//
// dst holds, per chunk, round and lane, the stage positions (entry 0, in
// bytes) of the contributions b = 0 .. n_local - 1 of the lane's unit, 0 past
// the last unit.  desc holds per chunk one word per lane of its groups,
// count | block << 4 | 4 row << 14 (block and row chunk-local; count 0 for a
// lane without a block), and long_desc two words per long block: block << 4 |
// 4 row << 14, and its first piece | contributions << 16.
constexpr int WAVE_SHORT = 8, WAVE_ROWS = 63, WAVE_BLOCKS = 1023, WAVE_GROUPS = 16, WAVE_STEP = 193;
struct WaveHead {
    int32_t row0, unit0, blk0, desc0; // first row, unit, pattern block and descriptor of the chunk
    int32_t n_rows, n_units, n_blocks, n_long;
    int32_t long0, long_base, n_groups, max_pieces; // first long block; most pieces of one
    uint8_t count[WAVE_GROUPS];                     // per group: largest count | smallest count << 4
};
struct WavePlanHost {
    std::vector<WaveHead> head; // every chunk holds at least one block
    std::vector<uint16_t> dst;
    std::vector<uint32_t> desc, long_desc;
    std::vector<int32_t> unused; // nodes outside the chunks: no element uses them
    int max_words = 0;           // stage words of the largest chunk
    double share = 0;            // of the chunks' lanes and rounds with a unit
};
// word_cap: stage words of a chunk of more than one node; value_size: bytes of
// an entry; word_limit: stage words of any chunk.  False when a row has more
// than 64 rounds (at most 2) units, WAVE_BLOCKS blocks or 64 long blocks, its
// stage exceeds word_limit or 64 KB, or the share is below least_share (found
// before the lanes are dealt, and as soon as the rows so far decide it).
bool make_wave_plan(const Pattern &pat, int n_local, const int32_t *elem_nodes, int rounds, int word_cap,
                    int value_size, WavePlanHost &out, int word_limit = 16384, double least_share = 0);

// The launch of the wavefront gather, by order, points and bytes of an entry.
// Units per lane:
constexpr int wave_rounds(int order, int n_quad) { return order == 1 && n_quad == 1 ? 2 : 1; }
// Stage words of a chunk of several nodes (three workgroups of four in a CU's
// LDS for FP32).  Fewer words leave lanes without a unit, more cost
// wavefronts: P2 mixed 363 us, with 2,496 words 387; P1 mixed 151, with 1,600
// words 160 and with 2,720 158; P1 FP64 (511,000 tets) 138, with 2,400 142.
constexpr int wave_words(int order, int value_size) { return order == 2 ? 2528 : value_size == 4 ? 2400 : 1600; }
// Wavefronts of a workgroup: they share the reference gradients alone.  P2
// mixed 363 us, with two 376, with one 431 (its waves then are the limit of
// workgroups per CU); of P2 FP64 one workgroup of eight fills the LDS.
constexpr int wave_group(int order, int value_size) { return order == 2 && value_size == 8 ? 8 : 4; }
// Bytes of the reference gradients that a workgroup keeps in LDS, and of its LDS
constexpr int wave_table(int order, int n_quad, int value_size) { return (order == 1 ? 4 : 10) * n_quad * 4 * value_size; }
constexpr int WAVE_LDS = 160 * 1024;
// The most words of a stage: every wavefront of the workgroup has one.  A chunk
// of one node takes what its blocks need, whatever wave_words says; a node of 52
// to 64 tets can need more than P2 FP64 has (2,540).
constexpr int wave_limit(int order, int n_quad, int value_size)
{
    return (WAVE_LDS - wave_table(order, n_quad, value_size)) / (wave_group(order, value_size) * value_size) / 4 * 4;
}
// The plan the library uses, of stages within wave_limit; max_words: the words
// of a stage as launched (a multiple of 4, and at least the gradient's staging
// of 3 doubles per unit).  False where make_wave_plan refuses.
bool plan_wave_gather(const Pattern &pat, int order, int n_quad, const int32_t *elem_nodes, int value_size, WavePlanHost &out,
                      double least_share = 0);
// The share from which the wavefront gather is the faster one on a large mesh
// (above 1: never), which wave_plan_ready passes as least_share; large_node: a
// node lies in more than 64 elements, so that the row-unit gather takes 256 units
// in a workgroup instead of 64.
//
// A chunk costs nearly the same whatever its lanes hold, and P1 rows of an
// unstructured mesh, with blocks of all counts, fill a stage with few units.
// E + G + H of 0.6 to 1.1 million P1 tets, wavefronts / the better row units, us:
//   one point FP64: lattice (share 0.73) 175 / 200, BCC points moved by 5 %
//   (0.68) 255 / 255, by 15 % (0.53) 292 / 259, by 25 % (0.30) 447 / 269, cubic
//   lattice points by 30 % (0.23) 586 / 291; with large nodes 267 / 307 (0.65),
//   303 / 315 (0.53), 460 / 331 (0.30), 604 / 381 (0.23)
//   one point FP32: lattice (0.93) 93 / 102, BCC 5 % (0.91) 129 / 128, 15 %
//   (0.84) 130 / 131 and with another numbering 144 / 136, 25 % (0.79) 143 / 135;
//   with large nodes 134 / 132 (0.91), 142 / 128 (0.84), 163 / 151 (0.81)
//   four points, FP64 and FP32: lattice 381 / 355 and 178 / 156, BCC 5 % 500 / 452
//   and 225 / 202
// At P2 the wavefronts are the faster ones throughout (161,000 tets of BCC points
// moved by 25 %: FP64 285 / 389, FP32 179 / 196).
constexpr double wave_share(int order, int n_quad, int value_size, bool large_node)
{
    if (order == 2) return 0;
    if (n_quad != 1) return 2;
    return value_size == 8 ? (large_node ? 0.55 : 0.7) : large_node ? 2 : 0.88;
}
double least_wave_share(const Pattern &pat, int order, int n_quad, int value_size);

// Chunks of consecutive outputs 0 .. n-1, output i gathering the
// contributions ptr[i] .. ptr[i+1]-1: a chunk holds at most cap
// contributions; c = chunk starts plus n.  False when one output alone has
// more than cap.
bool segment_chunks(const int32_t *ptr, int64_t n, int cap, std::vector<int32_t> &c);

// Row plan of the node-row gathers (k_gather_rows_seg): chunk[c] ..
// chunk[c+1]-1 are the rows of chunk c (at most ROW_SEG incidences);
// slot[c ROW_SEG + k] is the element-local vector index (node_inc code) of
// the chunk's k-th incidence, -1 past the last; rmeta[i] = q0 | count << 10,
// row i's first slot in its chunk and its incidence count.  False when a
// node has more than ROW_SEG incidences.
constexpr int ROW_SEG = 256;
struct RowPlanHost {
    std::vector<int32_t> chunk, slot, rmeta;
};
bool make_row_plan(const Pattern &pat, RowPlanHost &out);

// Per-contribution plan of the block and per-contribution factored gathers
// (k_gather_blocks_seg, k_gather_factored) for workgroups of gs threads:
// ptr[b] .. ptr[b+1]-1 are pattern block b's contributions (pattern order,
// n_blocks blocks); chunk[c] .. chunk[c+1]-1 are the blocks of chunk c (at
// most gs contributions), stored in the slots c gs .. (c+1) gs - 1 (-1 when
// unused) as words[k]; meta[b] = q0 | count << 10 | deg << 20 (first slot,
// count, the degree of b's row).  With keys (by element): each chunk's slots
// are ordered by keys[k] (ties in block order) and dst[c gs + i] is slot i's
// block-order position.  False when a block has more than gs contributions
// or a row more than 4095 blocks.
struct ContribPlanHost {
    std::vector<int32_t> chunk, slot, meta;
    std::vector<uint16_t> dst;
};
bool make_contrib_plan(const Pattern &pat, const std::vector<int32_t> &ptr, const std::vector<int32_t> &words,
                       const std::vector<int32_t> *keys, int gs, ContribPlanHost &out);

} // namespace pfgpu
