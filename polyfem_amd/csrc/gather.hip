// Wavefront gather of the factored route: the CSR values (and the gradient)
// from the element factor records, one wavefront per chunk of whole node rows
// (the plan and its layout are described at make_wave_plan in plans.hpp).
//
//   H_e(a, b) = (sum_q RG(q,a)^T G RG(q,b)) I + sum_q [cl_q k_a k_b^T + cc_q k_b k_a^T],
//   k_a = M_q RG(q, a),  G = w mu J^{-1} J^{-T} (the record's metric tail)
//
// Lane l forms the n_local blocks of unit l's row (a unit is a node
// incidence), the blocks' entries are staged in LDS at positions sorted by
// output block, the lanes add 64 output blocks at a time, and the sums leave
// through an LDS area in CSR order, so that consecutive lanes store
// consecutive blocks.  The row index m of the 3x3 blocks is the outer loop
// (three passes over the same registers): a third of the entries is staged
// at a time, which lets 12 wavefronts (FP32) share a CU's LDS.  A wavefront
// works alone, so no barrier ties the phases of different wavefronts together
// and one's formation runs beside another's sums.
//
// Formation, P2 at four points: the gradient of the edge (j, k) is
// 4 (lambda_j dlambda_k + lambda_k dlambda_j), that of vertex j
// (4 lambda_j - 1) dlambda_j, and lambda_j is HMS_B at one point and HMS_A at
// the other three.  So the entries of every column are combinations of the
// four vertex columns V_j(q) = la kappa_j^T + kappa_j lc^T + metric
// (kappa_j = M dlambda_j) summed over the points and at two points: about 710
// multiply-adds and additions per unit instead of the 1,104 multiply-adds of
// ten columns formed point by point.  (As a product A RG with A 9 x 12 per unit and
// the constant 12 x 10 table of reference gradients on the matrix cores,
// v_mfma_f32_4x4x1_16b, the vector ALUs keep 216 multiply-adds per unit, but
// the products, 68 us of them, did not overlap the rest: 411 us against
// 356 us for the 384,000-tet mesh below.)
//
// What bounds it: instruction issue and LDS latency of few wavefronts.  Of
// 340 us under the profiler (300 in a timed pass) for 384,000 P2 tets mixed,
// leaving out the sums takes 90 us off, the stores 72 and the gradient 20;
// formation alone needs 137 and its memory traffic about 150.  More wavefronts (16 instead of 12 per CU, by smaller
// chunks) gave nothing, since the smaller chunks leave lanes idle.
// E + G + H with this gather against the row-unit gather (64 units per workgroup,
// two threads per unit, a lane per piece of a block):
// 384,000 P2 tets NeoHookean mixed 450 -> 363 us, 44,600 P2 tets linear
// elasticity FP64 117 -> 87, 912,000 P1 tets mixed 162 -> 151, 511,000 P1 tets
// FP64 138 (lattice meshes; see gather_route in plain.hip for smaller ones and
// wave_share in plans.hpp for P1 meshes that do not take it).
#include "dispatch.hpp"
#include "factors.hpp"
#include "plans.hpp"

namespace pfgpu {

namespace {

template <typename T, int ORDER, int NQ> __constant__ RefTab<T, ORDER, NQ> c_ref = RefTab<T, ORDER, NQ>();

__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }

constexpr int N_XCD = 8;

// orders the LDS accesses of the wavefront's lanes (LDS serves a wavefront in order)
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the lane number as a value of this place: what is derived from it is
// computed here instead of being kept in registers over the whole kernel
// (spilled registers would put scratch loads, and with them a wait for all
// stores, into every pass)
__device__ __forceinline__ int lane_here()
{
    int l = int(threadIdx.x) & 63;
    asm volatile("" : "+v"(l));
    return l;
}

// what the sums and stores of a pass need of the chunk's head
struct Counts {
    int n_groups, n_long, long_base, max_pieces, nb, blk0, desc0;
    uint64_t cm_lo, cm_hi;
};

// a block's three summed entries and its row's first value, counted from the
// chunk's first and less three per block
template <typename T> struct alignas(4 * sizeof(T)) OutRow {
    T v[3];
    int32_t base;
};

// Groups whose descriptors are read ahead into registers, and 64-block stores
// of a pass issued whether or not the chunk has the blocks: with a fixed
// number of stores behind them, the loads of the next chunk are waited for
// without draining the stores.
constexpr int wave_ahead(int order) { return order == 2 ? 4 : 2; }

constexpr int wave_waves(int value_size) { return value_size == 4 ? 4 : 2; } // of a SIMD

template <typename T, int ORDER, int NQ, bool GRAD>
__global__ __launch_bounds__(64 * wave_group(ORDER, sizeof(T)), wave_waves(sizeof(T))) void k_gather_wave(
    int n_chunks, int last_unit, int words, const WaveHead *__restrict__ head, const int32_t *__restrict__ node_ptr,
    const int32_t *__restrict__ node_inc, const int32_t *__restrict__ brow_ptr, const uint32_t *__restrict__ dst,
    const uint32_t *__restrict__ desc, const uint32_t *__restrict__ long_desc, const T *__restrict__ rec,
    const T *__restrict__ gloc, T *__restrict__ values, double *__restrict__ grad)
{
    constexpr int NB = NLocal<ORDER>::value, R = fac_size(NQ), ROUNDS = wave_rounds(ORDER, NQ), AHEAD = wave_ahead(ORDER);
    constexpr int WAVES = wave_group(ORDER, sizeof(T));
    constexpr bool EDGES = ORDER == 2 && NQ == 4;
    constexpr int DW = NB / 2;
    // reference gradients of the lane's own node, [a][q] as (r0 r1 r2 0)
    __shared__ __align__(16) T srg[NB * NQ * 4];
    static_assert(sizeof(srg) == wave_table(ORDER, NQ, sizeof(T)));
    extern __shared__ __align__(32) unsigned char stages[];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    unsigned char *smem = stages + wave * words * int(sizeof(T)); // the wavefront's stage
    T *sv = reinterpret_cast<T *>(smem);
    double *sg = reinterpret_cast<double *>(smem);
    OutRow<T> *so = reinterpret_cast<OutRow<T> *>(smem);
    const RefTab<T, ORDER, NQ> &tb = c_ref<T, ORDER, NQ>;
    for (int k = threadIdx.x; k < NB * NQ * 4; k += 64 * WAVES) {
        const int a = k / (NQ * 4), q = k / 4 % NQ, l = k % 4;
        srg[k] = l < 3 ? tb.rg[(q * NB + a) * 3 + l] : T(0);
    }
    __syncthreads();
    const int per = (n_chunks + N_XCD - 1) / N_XCD, xcd = int(blockIdx.x % N_XCD);
    const int stride = int(gridDim.x / N_XCD) * WAVES, c_end = min(n_chunks, (xcd + 1) * per);
    int c = xcd * per + int(blockIdx.x / N_XCD) * WAVES + wave;
    if (c >= c_end) return;
    // Everything of a chunk that comes from memory.  The chunk after the
    // XCD's last is that one again.
    int row0, nr, nu, long0;
    Counts h;
    T r[ROUNDS][R], gl[ROUNDS][3];
    uint32_t dw[ROUNDS][DW], dd[AHEAD], ld[2];
    int a[ROUNDS];
    int32_t r0, deg, ru;
    // unit codes (e n_local + a), some other unit's past the chunk's last
    auto codes = [&](int cc, int32_t (&code)[ROUNDS]) {
        const int lane = lane_here();
        const int u0 = head[min(cc, c_end - 1)].unit0;
#pragma unroll
        for (int x = 0; x < ROUNDS; ++x) code[x] = node_inc[min(u0 + 64 * x + lane, last_unit)];
    };
    auto fetch = [&](int cc, const int32_t (&code)[ROUNDS]) {
        const int lane = lane_here();
        cc = min(cc, c_end - 1);
        const WaveHead &hd = head[cc];
        row0 = hd.row0, nr = hd.n_rows, nu = hd.n_units, long0 = hd.long0;
        const uint64_t *cw = reinterpret_cast<const uint64_t *>(hd.count);
        h = Counts{hd.n_groups, hd.n_long, hd.long_base, hd.max_pieces, hd.n_blocks, hd.blk0, hd.desc0, cw[0], cw[1]};
#pragma unroll
        for (int x = 0; x < ROUNDS; ++x) {
            const int e = code[x] / NB;
            a[x] = code[x] - e * NB;
            const T *rp = static_cast<const T *>(__builtin_assume_aligned(rec, 16)) + int64_t(e) * R;
#pragma unroll
            for (int i = 0; i < R; ++i) r[x][i] = rp[i];
#pragma unroll
            for (int p = 0; p < DW; ++p) dw[x][p] = dst[((int64_t(cc) * ROUNDS + x) * DW + p) * 64 + lane];
            if constexpr (GRAD)
#pragma unroll
                for (int d = 0; d < 3; ++d) gl[x][d] = gloc[int64_t(code[x]) * 3 + d];
        }
        const int rl = row0 + min(lane, nr);
        r0 = brow_ptr[rl];
        deg = brow_ptr[min(rl + 1, row0 + nr)] - r0;
        ru = node_ptr[rl] - hd.unit0;
    };
    // (long_desc is padded by one)
    auto descriptors = [&] {
        const int lane = lane_here();
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) dd[t] = desc[h.desc0 + 64 * min(t, max(h.n_groups - 1, 0)) + lane];
        const uint32_t *l = long_desc + 2 * int64_t(long0 + min(lane, max(h.n_long - 1, 0)));
        ld[0] = l[0], ld[1] = l[1];
    };
    int32_t code[ROUNDS];
    codes(c, code);
    fetch(c, code);
    descriptors();
    codes(c + stride, code);
    // the loads are complete here on the way in, so that inside the loop they
    // are waited for by the stores issued behind them
    __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0)
    for (; c < c_end; c += stride) {
        // ---- the gradient: one lane per (row, component), in unit order, FP64
        if constexpr (GRAD) {
            const int lane = lane_here();
#pragma unroll
            for (int x = 0; x < ROUNDS; ++x)
#pragma unroll
                for (int d = 0; d < 3; ++d) sg[(64 * x + lane) * 3 + d] = double(gl[x][d]);
            wave_order();
            for (int it = lane; it - lane < 3 * nr; it += 64) { // uniform over the wavefront
                const int row = min(it / 3, nr - 1), comp = it - it / 3 * 3;
                int u = __shfl(ru, row, 64);
                const int ue = __shfl(ru, row + 1, 64);
                double s = 0;
                for (; u + 4 <= ue; u += 4) {
                    const double *p = sg + u * 3 + comp;
                    const double g0 = p[0], g1 = p[3], g2 = p[6], g3 = p[9];
                    s += g0;
                    s += g1;
                    s += g2;
                    s += g3;
                }
                for (; u < ue; ++u) s += sg[u * 3 + comp];
                if (it < 3 * nr) grad[3 * int64_t(row0) + it] = s;
            }
            wave_order();
        }
        // ---- what the three passes share: cl k_a, cc k_a, G RG(q, a) per point
        T la[ROUNDS][NQ][3], lc[ROUNDS][NQ][3], ha[ROUNDS][NQ][3];
#pragma unroll
        for (int x = 0; x < ROUNDS; ++x) {
            const T *G6 = r[x] + 11 * NQ; // 00 11 22 01 02 12
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const T *M = r[x] + 9 * q, *ra = srg + (a[x] * NQ + q) * 4;
                const T ra0 = ra[0], ra1 = ra[1], ra2 = ra[2];
#pragma unroll
                for (int mm = 0; mm < 3; ++mm) {
                    const T ka = fma_t(M[mm * 3 + 2], ra2, fma_t(M[mm * 3 + 1], ra1, M[mm * 3] * ra0));
                    la[x][q][mm] = r[x][9 * NQ + q] * ka;
                    lc[x][q][mm] = r[x][10 * NQ + q] * ka;
                }
                ha[x][q][0] = fma_t(G6[4], ra2, fma_t(G6[3], ra1, G6[0] * ra0));
                ha[x][q][1] = fma_t(G6[5], ra2, fma_t(G6[1], ra1, G6[3] * ra0));
                ha[x][q][2] = fma_t(G6[2], ra2, fma_t(G6[5], ra1, G6[4] * ra0));
            }
        }
        // stage entry of contribution k of a round, in row part n
        auto stage = [&](int x, int k, int n) -> T & {
            const uint32_t at = k & 1 ? dw[x][k >> 1] >> 16 : dw[x][k >> 1] & 0xffffu;
            return *reinterpret_cast<T *>(smem + at + 64 * sizeof(T) * n);
        };
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            // ---- formation of the entries (m, 0 .. 2) into the stage
#pragma unroll
            for (int x = 0; x < ROUNDS; ++x) {
                if (64 * x + lane_here() >= nu) continue;
                if constexpr (EDGES) {
                    // vertex columns V_j(q) = la kappa_j^T + kappa_j lc^T + metric, kappa_j = M dlambda_j;
                    // lambda_j is HMS_B at one point (point 2 - (j - 1) for j = 1 .. 3, point 3 for
                    // j = 0) and HMS_A at the others
                    constexpr int EDGE_OF[4][4] = {{0, 4, 6, 7}, {4, 0, 5, 8}, {6, 5, 0, 9}, {7, 8, 9, 0}};
                    constexpr T va = T(4 * HMS_A - 1), vd = T(4 * (HMS_B - HMS_A)), ea = T(4 * HMS_A);
                    T ed[NB][3];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        T V[NQ][3];
#pragma unroll
                        for (int q = 0; q < NQ; ++q) {
                            const T *M = r[x] + 9 * q;
                            T kj[3];
#pragma unroll
                            for (int i = 0; i < 3; ++i) kj[i] = j ? M[i * 3 + j - 1] : -(M[i * 3] + M[i * 3 + 1] + M[i * 3 + 2]);
                            const T hj = j ? ha[x][q][j - 1] : -(ha[x][q][0] + ha[x][q][1] + ha[x][q][2]);
#pragma unroll
                            for (int n = 0; n < 3; ++n)
                                V[q][n] = fma_t(la[x][q][m], kj[n], m == n ? fma_t(kj[m], lc[x][q][n], hj) : kj[m] * lc[x][q][n]);
                        }
                        constexpr int peak[4] = {3, 2, 1, 0}; // the point where lambda_j is HMS_B
#pragma unroll
                        for (int n = 0; n < 3; ++n) {
                            const T S = (V[0][n] + V[1][n]) + (V[2][n] + V[3][n]);
                            stage(x, j, n) = fma_t(vd, V[peak[j]][n], va * S);
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (i != j) {
                                    // 4 lambda_i V_j summed over the points
                                    const T w = fma_t(vd, V[peak[i]][n], ea * S);
                                    T &o = ed[EDGE_OF[i][j]][n];
                                    if (i > j)
                                        o = w;
                                    else
                                        stage(x, EDGE_OF[i][j], n) = o + w;
                                }
                        }
                    }
                } else {
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        T v[3] = {T(0), T(0), T(0)};
#pragma unroll
                        for (int q = 0; q < NQ; ++q)
#pragma unroll
                            for (int l = 0; l < 3; ++l) {
                                const double rb = RG<ORDER, NQ>(q, b, l);
                                if (rb != 0.0) v[m] = fma_t(ha[x][q][l], T(rb), v[m]);
                            }
#pragma unroll
                        for (int q = 0; q < NQ; ++q) {
                            const T *M = r[x] + 9 * q;
                            T kb[3];
#pragma unroll
                            for (int mm = 0; mm < 3; ++mm) {
                                T s = T(0);
                                bool first = true;
#pragma unroll
                                for (int l = 0; l < 3; ++l) {
                                    const double rb = RG<ORDER, NQ>(q, b, l);
                                    if (rb != 0.0) {
                                        s = first ? M[mm * 3 + l] * T(rb) : fma_t(M[mm * 3 + l], T(rb), s);
                                        first = false;
                                    }
                                }
                                kb[mm] = s;
                            }
#pragma unroll
                            for (int n = 0; n < 3; ++n) v[n] = fma_t(kb[m], lc[x][q][n], fma_t(la[x][q][m], kb[n], v[n]));
                        }
#pragma unroll
                        for (int n = 0; n < 3; ++n) stage(x, b, n) = v[n];
                    }
                }
            }
            wave_order();
            // first value of row m of a node, less three per block before it,
            // counted from the chunk's first value
            const int32_t base = 6 * (r0 - h.blk0) + 3 * m * deg;
            // the rest of the pass needs the chunk's counts only: the next
            // chunk's data replaces the records
            const Counts now = h;
            if (m == 2) {
                fetch(c + stride, code);
                codes(c + 2 * stride, code);
            }
            auto row_base = [&](uint32_t d) { return __builtin_amdgcn_ds_bpermute(int(d >> 14) & 0xfc, base); };
            auto result = [&](uint32_t d) -> OutRow<T> & {
                return *reinterpret_cast<OutRow<T> *>(smem + (d & 0x3ff0u) * (sizeof(OutRow<T>) / 16));
            };
            // ---- short blocks, 64 at a time, contributions in unit order
            {
                uint64_t lo = now.cm_lo, hi = now.cm_hi;
                uint32_t ahead[AHEAD];
#pragma unroll
                for (int t = 0; t < AHEAD; ++t) ahead[t] = dd[t];
                const T *s = sv + lane_here();
                int word = 0;
                for (int t = 0; t < now.n_groups; ++t) {
                    const int most = int(lo & 15u), least = int(lo >> 4) & 15;
                    lo = (lo >> 8) | (hi << 56);
                    hi >>= 8;
                    if (t >= AHEAD) ahead[0] = desc[now.desc0 + 64 * t + lane_here()];
                    const uint32_t d = ahead[0];
#pragma unroll
                    for (int i = 0; i + 1 < AHEAD; ++i) ahead[i] = ahead[i + 1];
                    const int cnt = int(d & 15u);
                    const T *g = s + word;
                    // two contributions at a time
                    T v[3], p[3], q[3];
#pragma unroll
                    for (int n = 0; n < 3; ++n) v[n] = g[n * 64];
                    const int32_t ob = row_base(d);
                    if (most >= 2) {
#pragma unroll
                        for (int n = 0; n < 3; ++n) p[n] = g[WAVE_STEP + n * 64];
                        if (least >= 2) {
#pragma unroll
                            for (int n = 0; n < 3; ++n) v[n] += p[n];
                        } else {
#pragma unroll
                            for (int n = 0; n < 3; ++n) v[n] = cnt >= 2 ? v[n] + p[n] : v[n];
                        }
                    }
#pragma unroll
                    for (int k = 2; k < WAVE_SHORT; k += 2) {
                        if (k >= most) break;
#pragma unroll
                        for (int n = 0; n < 3; ++n) p[n] = g[WAVE_STEP * k + n * 64];
                        if (k + 1 < most) {
#pragma unroll
                            for (int n = 0; n < 3; ++n) q[n] = g[WAVE_STEP * (k + 1) + n * 64];
                            if (k + 2 <= least) {
#pragma unroll
                                for (int n = 0; n < 3; ++n) v[n] = (v[n] + p[n]) + q[n];
                            } else {
#pragma unroll
                                for (int n = 0; n < 3; ++n) {
                                    v[n] = k < cnt ? v[n] + p[n] : v[n];
                                    v[n] = k + 1 < cnt ? v[n] + q[n] : v[n];
                                }
                            }
                        } else {
#pragma unroll
                            for (int n = 0; n < 3; ++n) v[n] = k < cnt ? v[n] + p[n] : v[n];
                        }
                    }
                    wave_order();
                    if (cnt) result(d) = OutRow<T>{{v[0], v[1], v[2]}, ob};
                    word += 192 * most + 8;
                    // group 0 is read: the output area lies over it
                    if (t == 0) word = max(word, (4 * now.nb + 7) / 8 * 8);
                }
            }
            // ---- long blocks: a lane per (piece, entry), as many blocks at a
            // time as have room; then a block's first lane adds its pieces in order
            if (now.n_long) {
                const int step = 21 / now.max_pieces, lane = lane_here();
                for (int j = 0; j < now.n_long; j += step) {
                    const int x = min(lane / 3, 20), n = lane % 3, jb = x / now.max_pieces, piece = x - jb * now.max_pieces;
                    const int k = min(j + jb, now.n_long - 1);
                    const uint32_t d = __shfl(ld[0], k, 64), w = __shfl(ld[1], k, 64);
                    const int left = int(w >> 16) - WAVE_SHORT * piece, at = int(w & 0xffffu) + (left > 0 ? piece : 0);
                    const T *s = sv + now.long_base + at / 8 * 192 + n * 64 + at % 8 * 8;
                    T v = s[0];
#pragma unroll
                    for (int i = 1; i < WAVE_SHORT; ++i) {
                        const T p = s[i];
                        v = i < left ? v + p : v;
                    }
                    T tot = v;
                    for (int i = 1; i < now.max_pieces; ++i) {
                        const T p = __shfl(v, lane + 3 * i, 64);
                        tot = WAVE_SHORT * i < left ? tot + p : tot;
                    }
                    const int32_t ob = row_base(d);
                    wave_order();
                    if (lane < 63 && piece == 0 && jb < step && j + jb < now.n_long) {
                        result(d).v[n] = tot;
                        if (n == 0) result(d).base = ob;
                    }
                }
            }
            wave_order();
            if (m == 2) descriptors(); // of the next chunk
            // ---- row m of every block, consecutive lanes on consecutive
            // blocks (past the last one, the last again)
            T *const out = values + 9 * int64_t(now.blk0);
            const int lane = lane_here();
            auto store = [&](int k) {
                const OutRow<T> o = so[k];
                T *p = out + uint32_t(o.base + 3 * k);
#pragma unroll
                for (int n = 0; n < 3; ++n) {
                    // past the caches where a lane's row entries are 24 bytes
                    // (P1 FP64, 511,000 tets: 138 us against 163); with 12 the
                    // caches have to merge the lines (P1 mixed 160 against 166)
                    if constexpr (sizeof(T) == 8)
                        __builtin_nontemporal_store(o.v[n], p + n);
                    else
                        p[n] = o.v[n];
                }
            };
#pragma unroll
            for (int t = 0; t < AHEAD; ++t) store(min(64 * t + lane, now.nb - 1));
            for (int k = 64 * AHEAD + lane; k < now.nb; k += 64) store(k);
            wave_order();
        }
    }
}

// the gradient of nodes no element uses
__global__ __launch_bounds__(BLOCK) void k_zero_nodes(int n, const int32_t *__restrict__ nodes, double *__restrict__ grad)
{
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i < n)
        for (int d = 0; d < 3; ++d) grad[3 * int64_t(nodes[i]) + d] = 0.0;
}

} // namespace

// the wavefront plan of the handle; false when a node has too many incident
// elements for one chunk, or blocks for a stage that the workgroup's LDS holds,
// or the chunks would have too few units (wave_share; the row-unit gather then
// serves the handle)
bool wave_plan_ready(Handle &h)
{
    if (h.wave_plan.state == 0) {
        WavePlanHost w;
        const double least = least_wave_share(h.pat, h.order, h.n_quad, int(h.value_size()));
        if (9 * h.pat.n_blocks >= (int64_t(1) << 31) || least > 1 ||
            !plan_wave_gather(h.pat, h.order, h.n_quad, h.h_elem_nodes.data(), int(h.value_size()), w, least)) {
            h.wave_plan.state = -1;
        } else {
            h.wave_plan.head = upload(w.head, h.stream);
            h.wave_plan.dst = upload(w.dst, h.stream);
            // one group and one long block more: read ahead, not used
            w.desc.resize(w.desc.size() + 64);
            w.long_desc.resize(w.long_desc.size() + 2);
            h.wave_plan.desc = upload(w.desc, h.stream);
            h.wave_plan.long_desc = upload(w.long_desc, h.stream);
            h.wave_plan.unused = upload(w.unused, h.stream);
            h.wave_plan.n_unused = int(w.unused.size());
            h.wave_plan.n_chunks = int(w.head.size());
            h.wave_plan.words = w.max_words;
            if (!h.brow_ptr.get()) h.brow_ptr = upload(h.pat.brow_ptr, h.stream);
            h.wave_plan.state = 1;
        }
    }
    return h.wave_plan.state == 1;
}

// the CSR values (and, with gloc, the gradient) from the factor records in h.fac_rec
void wave_gather(Handle &h, const void *gloc, double *g, void *values)
{
    WavePlan &p = h.wave_plan;
    dispatch<true>(h, [&]<typename T, int O, int Q, int M>() {
        if constexpr ((M == MAT_NH || M == MAT_LE) && wave_share(O, Q, sizeof(T), false) <= 1) {
            auto go = [&]<bool GRAD>() {
                constexpr int WAVES = wave_group(O, sizeof(T));
                auto kern = k_gather_wave<T, O, Q, GRAD>;
                const int lds = WAVES * p.words * int(sizeof(T));
                unsigned &grid = GRAD ? p.grid_grad : p.grid;
                if (grid == 0) {
                    // the function's limit, not the handle's: one value that every plan fits
                    PF_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                               WAVE_LDS - wave_table(O, Q, int(sizeof(T)))));
                    if (h.n_cu == 0) PF_HIP(hipDeviceGetAttribute(&h.n_cu, hipDeviceAttributeMultiprocessorCount, h.device));
                    int per_cu = 0;
                    PF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, 64 * WAVES, size_t(lds)));
                    const int n = std::max(1, h.n_cu) * std::max(1, per_cu);
                    const int most = ((p.n_chunks + N_XCD - 1) / N_XCD + WAVES - 1) / WAVES;
                    grid = unsigned(std::min(most, (n + N_XCD - 1) / N_XCD) * N_XCD);
                }
                kern<<<grid, 64 * WAVES, lds, h.stream>>>(p.n_chunks, int(h.pat.node_inc.size()) - 1, p.words, p.head.as<WaveHead>(), h.node_ptr.as<int32_t>(),
                                                  h.node_inc.as<int32_t>(), h.brow_ptr.as<int32_t>(), p.dst.as<uint32_t>(),
                                                  p.desc.as<uint32_t>(), p.long_desc.as<uint32_t>(), h.fac_rec.as<T>(), static_cast<const T *>(gloc),
                                                  static_cast<T *>(values), g);
            };
            if (gloc) {
                go.template operator()<true>();
                if (p.n_unused)
                    k_zero_nodes<<<grid_for(p.n_unused), BLOCK, 0, h.stream>>>(p.n_unused, p.unused.as<int32_t>(), g);
            } else {
                go.template operator()<false>();
            }
        } else {
            fail(PFGPU_ERR_INVALID_STATE, "the wavefront gather does not cover this rule or material");
        }
    });
    PF_LAUNCH_CHECK();
}

} // namespace pfgpu
