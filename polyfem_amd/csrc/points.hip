// Element Hessians of the materials outside the factored form (SaintVenant,
// FixedCorotational, MooneyRivlin), in k_hessian's 64-element tiles.
//
// The tangent of each material is a sum of outer products of a few vectors
// per node and quadrature point, each a linear map of the node's reference
// gradient: with per-point 3x3 maps in registers, a block costs a few maps
// of the column's gradient and the outer products (57 to 105 FP32
// instructions per block and point).  What bounds the kernel is the register
// footprint of those maps, so the points of an element are dealt to LPE = 2
// or 4 neighbouring lanes (one lane for the one-point rule): a lane keeps the
// maps of ceil(NQ / LPE) points only, a wavefront covers 64 / LPE elements, and a
// block's partial sums meet in one permute and one addition in LDS.
//
// 45,360 P2 MooneyRivlin tets, mixed precision: 48 us; one thread per element
// with the directional stress derivative formed again per block column and
// point took 2,149 us.
#include "dispatch.hpp"

namespace pfgpu {

namespace {

// v of the neighbouring lane (lanes 1 0 3 2 of a quad)
__device__ __forceinline__ float pair_swap(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, true));
}
__device__ __forceinline__ double pair_swap(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xb1, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xb1, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// out = A r (3x3)
template <typename T> __device__ __forceinline__ void map3(const T *A, const T *r, T *out)
{
#pragma unroll
    for (int i = 0; i < 3; ++i) out[i] = A[3 * i] * r[0] + A[3 * i + 1] * r[1] + A[3 * i + 2] * r[2];
}
// out = A r for symmetric A (00 11 22 01 02 12)
template <typename T> __device__ __forceinline__ void map_sym(const T *A, const T *r, T *out)
{
    out[0] = A[0] * r[0] + A[3] * r[1] + A[4] * r[2];
    out[1] = A[3] * r[0] + A[1] * r[1] + A[5] * r[2];
    out[2] = A[4] * r[0] + A[5] * r[1] + A[2] * r[2];
}
template <typename T> __device__ __forceinline__ T dot3(const T *a, const T *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
// v += a b^T
template <typename T> __device__ __forceinline__ void outer_add(const T *a, const T *b, T *v)
{
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int n = 0; n < 3; ++n) v[3 * m + n] += a[m] * b[n];
}
// out[m][k] = sum_c A[m][c] jit[k][c]: the map from reference gradients to A G
template <typename T> __device__ __forceinline__ void to_reference(const T *A, const T *jit, T *out)
{
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int k = 0; k < 3; ++k) out[3 * m + k] = A[3 * m] * jit[3 * k] + A[3 * m + 1] * jit[3 * k + 1] + A[3 * m + 2] * jit[3 * k + 2];
}

// One quadrature point's form: init() from the kinematics, row() what the
// blocks of a row a share, block() the contribution to block (a, b).  ra, rb
// are reference gradients, g6 the metric jit jit^T, w = det J x the weight.
template <typename T, int MAT> struct PointForm;

// H_ab = (G_a^T S G_b) I + mu (G_a . G_b) F F^T + lambda k_a k_b^T + mu k_b k_a^T, k = F G
template <typename T> struct PointForm<T, MAT_SV> {
    T M[9], sg[6], ff[6], cl, cc;
    struct Row {
        T us[3], ug[3], la[3], lc[3];
    };
    __device__ __forceinline__ void init(const Kin<T> &k, const T *jit, T lam, T mu, T, T w)
    {
        hess_qp<T, MAT_SV>(k, jit, lam, mu, w, M, cl, cc);
        sv_extra(k.H, jit, lam, mu, w, sg, ff);
    }
    __device__ __forceinline__ void row(const T *g6, const T *ra, Row &r) const
    {
        T ka[3];
        map3(M, ra, ka);
        map_sym(sg, ra, r.us);
        map_sym(g6, ra, r.ug);
#pragma unroll
        for (int i = 0; i < 3; ++i) r.la[i] = cl * ka[i], r.lc[i] = cc * ka[i];
    }
    __device__ __forceinline__ void block(const Row &r, const T *rb, T *v) const
    {
        T kb[3];
        map3(M, rb, kb);
        const T gd = dot3(r.us, rb), gq = dot3(r.ug, rb);
        const int sym[9] = {0, 3, 4, 3, 1, 5, 4, 5, 2};
#pragma unroll
        for (int i = 0; i < 9; ++i) v[i] += gq * ff[sym[i]] + (i % 4 == 0 ? gd : T(0));
        outer_add(r.la, kb, v);
        outer_add(kb, r.lc, v);
    }
};

// H_ab = 2 mu (G_a . G_b) I + cl k_a k_b^T + cc k_b k_a^T - 2 mu (G_a x r_m)^T K^{-1} (G_b x r_n),
// k = F^{-T} G, r_m the rows of R.  With g = R G the last term is
// (g_a x e_m)^T (R K^{-1} R^T) (g_b x e_n), whose cross products are signed
// permutations of g.
template <typename T> struct PointForm<T, MAT_FC> {
    T M[9], Mg[9], Kt[6], cl, cc, cm;
    struct Row {
        T us[3], la[3], lc[3], t[9];
    };
    __device__ __forceinline__ void init(const Kin<T> &k, const T *jit, T lam, T mu, T, T w)
    {
        hess_qp<T, MAT_FC>(k, jit, lam, mu, w, M, cl, cc);
        cm = T(2) * mu * w;
        FcKin<T> f;
        fc_kinematics(k.H, f);
        T R[9], RK[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) R[i] = f.Q[i] + (i % 4 == 0 ? T(1) : T(0));
        to_reference(R, jit, Mg);
        const T s = -cm;
        const T K[9] = {s * f.Ki6[0], s * f.Ki6[3], s * f.Ki6[4], s * f.Ki6[3], s * f.Ki6[1],
                        s * f.Ki6[5], s * f.Ki6[4], s * f.Ki6[5], s * f.Ki6[2]};
        mul3(R, K, RK);
        auto rk = [&](int i, int j) { return RK[3 * i] * R[3 * j] + RK[3 * i + 1] * R[3 * j + 1] + RK[3 * i + 2] * R[3 * j + 2]; };
        Kt[0] = rk(0, 0), Kt[1] = rk(1, 1), Kt[2] = rk(2, 2), Kt[3] = rk(0, 1), Kt[4] = rk(0, 2), Kt[5] = rk(1, 2);
    }
    __device__ __forceinline__ void row(const T *g6, const T *ra, Row &r) const
    {
        T ka[3], g[3];
        map3(M, ra, ka);
        map3(Mg, ra, g);
        map_sym(g6, ra, r.us);
#pragma unroll
        for (int i = 0; i < 3; ++i) r.us[i] *= cm, r.la[i] = cl * ka[i], r.lc[i] = cc * ka[i];
        // t[m] = Kt (g x e_m)
        const T c[3][3] = {{T(0), g[2], -g[1]}, {-g[2], T(0), g[0]}, {g[1], -g[0], T(0)}};
#pragma unroll
        for (int m = 0; m < 3; ++m) map_sym(Kt, c[m], r.t + 3 * m);
    }
    __device__ __forceinline__ void block(const Row &r, const T *rb, T *v) const
    {
        T kb[3], g[3];
        map3(M, rb, kb);
        map3(Mg, rb, g);
        const T gd = dot3(r.us, rb);
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const T *t = r.t + 3 * m;
            v[3 * m] += t[1] * g[2] - t[2] * g[1];
            v[3 * m + 1] += t[2] * g[0] - t[0] * g[2];
            v[3 * m + 2] += t[0] * g[1] - t[1] * g[0];
            v[4 * m] += gd;
        }
        outer_add(r.la, kb, v);
        outer_add(kb, r.lc, v);
    }
};

// MooneyRivlin: the columns dP[e_n G_b^T] G_a of mr_dstress with k = F^{-T} G,
// f = F G, h = B F G (a = c1 J^{-2/3} w, b = c2 J^{-4/3} w):
//   H_ab = [(2a + 2b I1) (G_a . G_b) - 2b (f_a . f_b)] I - 2b (G_a . G_b) B
//        + p_a f_b^T + z_a k_b^T + (8/3 b) k_a h_b^T + s4 k_b k_a^T - 2b f_b f_a^T,
//   p_a = 4b f_a - (4/3 a + 8/3 b I1) k_a,  z_a = (kappa w) k_a - (2/3 a R1 + 4/3 b Q2) G_a,
//   s4 = 2/3 a I1 + 4/3 b I2 - kappa w ln J.
template <typename T> struct PointForm<T, MAT_MR> {
    T Mk[9], Mf[9], Mh[9], Mz[9], iso[6], Bb[6], b, c, s4;
    struct Row {
        T us[3], ug[3], p[3], z[3], kh[3], ks[3], fs[3];
    };
    __device__ __forceinline__ void init(const Kin<T> &k, const T *jit, T c1, T c2, T kk, T w)
    {
        MrKin<T> r;
        mr_kinematics(k, r);
        T R1[9], Q2[9];
        mr_brackets(k, r, R1, Q2);
        const T *H = k.H;
        const T F[9] = {T(1) + H[0], H[1], H[2], H[3], T(1) + H[4], H[5], H[6], H[7], T(1) + H[8]};
        const T B[9] = {T(1) + r.S[0], r.S[1], r.S[2], r.S[3], T(1) + r.S[4], r.S[5], r.S[6], r.S[7], T(1) + r.S[8]};
        const T I1 = T(3) + r.i1, I2 = T(3) + r.i2;
        const T a = w * c1 * (T(1) + r.ea), kw = w * kk;
        b = w * c2 * (T(1) + r.eb);
        c = -(T(4.0 / 3.0) * a + T(8.0 / 3.0) * b * I1);
        s4 = T(2.0 / 3.0) * a * I1 + T(4.0 / 3.0) * b * I2 - kw * k.lnJ;
        T BF[9], Z[9];
        mul3(B, F, BF);
#pragma unroll
        for (int i = 0; i < 9; ++i) Z[i] = kw * k.FmT[i] - (T(2.0 / 3.0) * a * R1[i] + T(4.0 / 3.0) * b * Q2[i]);
        to_reference(k.FmT, jit, Mk);
        to_reference(F, jit, Mf);
        to_reference(BF, jit, Mh);
        to_reference(Z, jit, Mz);
        // (2a + 2b I1) jit jit^T - 2b (F jit^T)^T (F jit^T), reference indices
        T g6[6];
        metric(jit, g6);
        const int kk6[6] = {0, 1, 2, 0, 0, 1}, ll6[6] = {0, 1, 2, 1, 2, 2}, s9[6] = {0, 4, 8, 1, 2, 5};
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const T f = Mf[kk6[i]] * Mf[ll6[i]] + Mf[3 + kk6[i]] * Mf[3 + ll6[i]] + Mf[6 + kk6[i]] * Mf[6 + ll6[i]];
            iso[i] = (T(2) * a + T(2) * b * I1) * g6[i] - T(2) * b * f;
            Bb[i] = -T(2) * b * B[s9[i]];
        }
    }
    __device__ __forceinline__ void row(const T *g6, const T *ra, Row &r) const
    {
        T ka[3], fa[3];
        map3(Mk, ra, ka);
        map3(Mf, ra, fa);
        map3(Mz, ra, r.z);
        map_sym(iso, ra, r.us);
        map_sym(g6, ra, r.ug);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            r.p[i] = c * ka[i] + T(4) * b * fa[i];
            r.kh[i] = T(8.0 / 3.0) * b * ka[i];
            r.ks[i] = s4 * ka[i];
            r.fs[i] = -T(2) * b * fa[i];
        }
    }
    __device__ __forceinline__ void block(const Row &r, const T *rb, T *v) const
    {
        T kb[3], fb[3], hb[3];
        map3(Mk, rb, kb);
        map3(Mf, rb, fb);
        map3(Mh, rb, hb);
        const T gd = dot3(r.us, rb), gq = dot3(r.ug, rb);
        const int sym[9] = {0, 3, 4, 3, 1, 5, 4, 5, 2};
#pragma unroll
        for (int i = 0; i < 9; ++i) v[i] += gq * Bb[sym[i]] + (i % 4 == 0 ? gd : T(0));
        outer_add(r.p, fb, v);
        outer_add(r.z, kb, v);
        outer_add(r.kh, hb, v);
        outer_add(kb, r.ks, v);
        outer_add(fb, r.fs, v);
    }
};

// Lanes per element.  SaintVenant in FP32 at four points has the smallest
// form: two lanes with two points each still fit four wavefronts per SIMD, and
// the row and reduction work per element is shared by fewer lanes (P2 Hessian
// with its gather, mixed: 384,000 tets 802 us against 840 us with four lanes
// and 808 us with one; 10,368 tets 46 us against 43 us and 69 us).
//
// On large P1 meshes (from 16,384 elements) two lanes are the better ones for
// six points, of which four lanes leave a quarter idle, and for SaintVenant's four
// points in FP64 too: with ten blocks per element the points' forms are most of the
// work, and there are elements enough.  843,648 P1 tets, Hessian with its gather,
// two / four lanes, us: SaintVenant six points FP64 536 / 551, FP32 278 / 310,
// four points FP64 435 / 450 (one thread per element with the form of this material
// alone: 502, 267 and 402); FixedCorotational 995 / 1,274 and 588 / 686,
// MooneyRivlin 766 / 941 and 354 / 444; 24,576 tets: SaintVenant 27.1 / 30.1, 19.6 /
// 19.4 and 25.3 / 26.3; 1,296 tets 14.8 / 13.3, 13.2 / 11.9 and 13.4 / 12.1.
constexpr int POINTS_LARGE = 16384;
template <typename T, int MAT> constexpr int points_lanes(int order, int nq, bool large)
{
    if (nq == 1) return 1;
    if (MAT == MAT_SV && sizeof(T) == 4 && nq == 4) return 2;
    return order == 1 && large && (nq == 6 || (MAT == MAT_SV && nq == 4)) ? 2 : 4;
}

// hloc as k_hessian writes it: block s of element e at
// (((e / 64) NBLK + s) 64 + e % 64) 9.  Lane l of a wavefront takes element
// l / LPE of the wavefront's 64 / LPE and the points l % LPE + LPE j; a lane
// past the rule's last point carries weight zero.  A block of the wavefront's
// elements is one contiguous run: each pair of lanes adds its partial sums,
// the pairs' 9 values are staged in LDS, and the lanes that store the run add
// the two pairs of an element (finishing the sum by quad permutes instead
// costs 20 more VALU instructions per block, 25 % of the kernel's).
template <typename T, int ORDER, int NQ, int MAT, int LPE>
__global__ __launch_bounds__(BLOCK) void k_hessian_points(DevMesh<T> m, const double *__restrict__ x, T *__restrict__ hloc)
{
    constexpr int NB = NLocal<ORDER>::value, NBLK = NB * (NB + 1) / 2;
    constexpr int QPL = (NQ + LPE - 1) / LPE, EPW = 64 / LPE, RUN = EPW * 9;
    constexpr int HALVES = LPE == 4 ? 2 : 1, NOUT = (RUN + 63) / 64;
    __shared__ __align__(16) T stage[BLOCK / 64][RUN * HALVES];
    // reference gradients (r0 r1 r2) and weight per (point, node)
    __shared__ __align__(16) T rg[NQ * NB * 4];
    for (int i = threadIdx.x; i < NQ * NB; i += BLOCK) {
        const int q = i / NB, a = i - q * NB;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            rg[4 * i + k] = T(ref_grad<ORDER>(quad_point(NQ, q, 0), quad_point(NQ, q, 1), quad_point(NQ, q, 2), a, k));
        rg[4 * i + 3] = T(quad_weight(NQ, q));
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ql = lane % LPE;
    const int e0 = (int(blockIdx.x) * (BLOCK / 64) + wv) * EPW; // the wavefront's first element
    if (e0 >= m.n_elements) return;                             // uniform over the wavefront
    // lanes past the last element compute on element 0; their blocks land in
    // the last tile's padding
    const int e = e0 + lane / LPE < m.n_elements ? e0 + lane / LPE : 0;
    PointForm<T, MAT> form[QPL];
    T g6[6];
    int qs[QPL];
    {
        Elem<T, ORDER, NQ> el;
        load_geometry(m, e, el);
        gather(m, e, x, el.U);
        metric(el.jit, g6);
#pragma unroll
        for (int j = 0; j < QPL; ++j) {
            const int q = ql + LPE * j;
            qs[j] = q < NQ ? q : 0;
            const T *r = rg + 4 * NB * qs[j];
            const T w = q < NQ ? el.det * r[3] : T(0);
            Kin<T> k;
            T A[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) A[i] = T(0);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int c = 0; c < 3; ++c) A[3 * d + c] += el.U[b][d] * r[4 * b + c];
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    k.H[3 * d + c] = A[3 * d] * el.jit[c] + A[3 * d + 1] * el.jit[3 + c] + A[3 * d + 2] * el.jit[6 + c];
            if (MAT != MAT_SV) kinematics(k);
            form[j].init(k, el.jit, el.lam, el.mu, el.p3, w);
        }
    }
    T *st = stage[wv];
    // output i = 9 element + entry of a block's run; the element's first pair
    int at[NOUT];
#pragma unroll
    for (int j = 0; j < NOUT; ++j) {
        const int i = 64 * j + lane, le = i / 9;
        at[j] = HALVES * 9 * le + (i - 9 * le);
    }
    T *out = hloc + int64_t(e0 / 64) * NBLK * 576 + (e0 % 64) * 9;
#pragma unroll 1
    for (int a = 0; a < NB; ++a) {
        typename PointForm<T, MAT>::Row row[QPL];
#pragma unroll
        for (int j = 0; j < QPL; ++j) form[j].row(g6, rg + 4 * (NB * qs[j] + a), row[j]);
#pragma unroll 1
        for (int b = a; b < NB; ++b) {
            T v[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) v[i] = T(0);
#pragma unroll
            for (int j = 0; j < QPL; ++j) form[j].block(row[j], rg + 4 * (NB * qs[j] + b), v);
            if constexpr (LPE >= 2)
#pragma unroll
                for (int i = 0; i < 9; ++i) v[i] += pair_swap(v[i]);
            if (LPE == 1 || lane % 2 == 0) {
                T *s = st + (LPE == 1 ? lane : lane / 2) * 9;
#pragma unroll
                for (int i = 0; i < 9; ++i) s[i] = v[i];
            }
            __builtin_amdgcn_wave_barrier();
            const int s = a * NB - a * (a - 1) / 2 + (b - a);
#pragma unroll
            for (int j = 0; j < NOUT; ++j)
                if (RUN % 64 == 0 || j < NOUT - 1 || lane < RUN % 64) {
                    T o = st[at[j]];
                    if constexpr (HALVES == 2) o += st[at[j] + 9];
                    out[s * 576 + 64 * j + lane] = o;
                }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

} // namespace

void points_hessian(Handle &h, const double *x, void *hloc)
{
    dispatch(h, [&]<typename T, int O, int Q, int M>() {
        if constexpr (M == MAT_SV || M == MAT_FC || M == MAT_MR) {
            auto go = [&]<int LPE>() {
                k_hessian_points<T, O, Q, M, LPE><<<grid_for(int64_t(h.n_elements) * LPE), BLOCK, 0, h.stream>>>(h.mesh<T>(), x,
                                                                                                             static_cast<T *>(hloc));
            };
            if (h.n_elements < POINTS_LARGE)
                go.template operator()<points_lanes<T, M>(O, Q, false)>();
            else
                go.template operator()<points_lanes<T, M>(O, Q, true)>();
        } else {
            fail(PFGPU_ERR_INVALID_STATE, "the point-parallel Hessian covers SaintVenant, FixedCorotational and MooneyRivlin");
        }
    });
    PF_LAUNCH_CHECK();
}

} // namespace pfgpu
