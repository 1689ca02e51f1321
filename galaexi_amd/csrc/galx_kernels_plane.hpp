// galx_kernels_plane.hpp -- stage kernels in which a workgroup takes a few k-planes of an element instead of the whole
// element: for degrees whose elements have more nodes than a workgroup has threads (N >= GALX_PLANE_DEGREE, 10), and
// for meshes of few elements, where one workgroup per element leaves most of the chip idle (use_planes).
//   k_vol_plane : BR1 gradients, the viscous and split (or weak Euler) volume terms except the D_Hat contraction along
//                 k, and the face nodes' normal viscous fluxes (vtr).  Everything along i and j stays in the planes of
//                 the workgroup; along k a node reads its own column of U and Ja^3 (each value once: staged in LDS it
//                 would be used once too), the neighbouring nodes' columns coalesced, from the L2 that the element's
//                 other planes read through as well (plane_block).
//   k_upd_plane : the D_Hat contraction along k from the contravariant fluxes f_3 that k_vol_plane left in the
//                 workspace, the face fluxes, -sJ, the register update and the next traces.
// The gradients are formed once per stage, where k_lift and k_rhs form the surface nodes' twice; the price is the
// workspace, 9 (split) or 10 (weak) values per node written and read once, and each column read by every plane.
// On small meshes both kernels are bound by the latency of one workgroup's instruction stream, not by bytes: k_vol_plane
// issues 2272 VALU and 291 LDS instructions a wave at N = 11 (2^3 elements, 15.3 us, 0.3 TB/s, VALU busy 4 %, occupancy
// 2 %), 1666 and 220 at N = 7 (4^3, 13.2 us, 0.8 TB/s, 6 %, 3 %); loads issued ahead of the state changed nothing and cost
// spills.  Measured on MI355X, FP64, us per stage of a run, launches included, with one workgroup per element (k_lift +
// k_rhs) and with planes, split LF, weak Roe and split RoeEntropyFix:
//   N = 4: 2^3 16.6 -> 16.2, 15.3 -> 15.5, 17.1 -> 17.5; 4^3 16.7 -> 15.5, 15.3 -> 15.1, 17.1 -> 16.9;
//          5^3 16.9 -> 17.3, 15.6 -> 16.7, 17.4 -> 18.5; 6^3 17.5 -> 18.0, 16.0 -> 17.1, 17.9 -> 19.2
//   N = 5: 2^3 19.8 -> 16.4, 17.1 -> 15.0, 20.3 -> 17.5; 5^3 20.4 -> 19.7, 17.6 -> 17.2, 20.8 -> 20.6;
//          6^3 21.1 -> 22.0, 18.5 -> 20.5, 21.6 -> 23.3
//   N = 6: 4^3 22.6 -> 18.4, 19.9 -> 17.0, 23.7 -> 19.6; 5^3 23.5 -> 21.7, 20.7 -> 20.5, 24.6 -> 22.7;
//          6^3 24.9 -> 24.3, 21.9 -> 23.1, 25.9 -> 26.1
//   N = 7: 2^3 25.4 -> 17.5, 22.2 -> 16.1, 26.8 -> 18.7; 5^3 26.9 -> 23.0, 23.7 -> 21.4, 28.5 -> 24.5;
//          6^3 28.4 -> 30.0, 25.0 -> 28.3, 29.7 -> 32.6
//   N = 8: 4^3 33.1 -> 22.8, 27.0 -> 20.6, 32.7 -> 23.8; 5^3 35.0 -> 30.2, 28.4 -> 27.3, 34.2 -> 31.7;
//          6^3 37.3 -> 39.4, 30.1 -> 35.6, 36.4 -> 40.7
//   N = 9: 2^3 37.6 -> 20.1, 30.9 -> 17.3, 39.2 -> 24.6; 4^3 38.3 -> 26.4, 31.6 -> 22.6, 39.9 -> 30.6;
//          5^3 40.1 -> 35.8, 33.3 -> 30.3, 41.8 -> 44.3; 6^3 43.0 -> 55.2, 35.6 -> 47.6, 44.5 -> 74.2
// On meshes that fill the chip they lose (both kernels: N = 8, 12^3 247 -> 275, N = 9, 12^3 347 -> 416 us).  For N >= 10
// they replaced kernels with all work arrays in HBM (N = 11, 2^3, split, RoeEntropyFix 303 -> 24 us).
#pragma once
#include "galx_kernels.hpp"

#ifndef GALX_PLANE_DEGREE
#define GALX_PLANE_DEGREE 10
#endif

namespace galx {

template <int N>
struct Pl {
    static constexpr int n = N + 1, n2 = n * n, n3 = n2 * n;
    // planes per workgroup: one plane is 25 of 64 lanes at N = 4 and 81 of 128 at N = 8, two and three are 50 of 64 and
    // 243 of 256 (at N = 8 one plane measured 29 against 27 us on 4^3 elements).  N = 5, 36 of 64 lanes, has been measured
    // with one plane only; the other degrees fill three quarters of their lanes or more
    static constexpr int planes = N == 4 ? 2 : (N == 8 ? 3 : 1);
    static constexpr int block = (planes * n2 + 63) / 64 * 64;
    static constexpr int groups = (n + planes - 1) / planes;  // workgroups per element
    static constexpr int ws = 10 * n3;  // workspace values per element: [5] volume terms, [5] contravariant flux f_3
};

// FP64 meshes of at most four planes a CU take the plane kernels from N = 4 on: one line for all degrees, near which the two
// forms cross (see the figures above).  It is not each degree's own: the planes still win beyond it at N = 8 and 9 (5^3
// elements, up to 14 %, but not with RoeEntropyFix at N = 9), and lose up to 7 % below it at N = 4 (5^3).  The mixed form
// keeps its one-element kernels and with them its FP32 rounding; it takes the planes from N = 10 on, in a library built for
// such mixed degrees (Ut at N = 11 5.5e-6 split LF, 3.8e-6 weak Roe from the FP64 oracle).
template <int N, typename T>
__host__ constexpr bool use_planes(int nElems)
{
    return N >= GALX_PLANE_DEGREE || (sizeof(T) == 8 && N >= 4 && (long)nElems * (N + 1) <= 4 * CUS);
}

// workgroups are dealt to the 8 XCDs in turn: workgroup x takes block (x % 8) * per + x / 8 of `count` blocks, so that
// each XCD works on one contiguous range and the planes of an element read its columns through one L2.  Grid: 8 * per
// with per = ceil(count / 8); -1 beyond the end.
__host__ __device__ inline int plane_per_xcd(int count) { return (count + 7) / 8; }

__device__ __forceinline__ int plane_block(int count)
{
    const int b = (blockIdx.x & 7) * plane_per_xcd(count) + (blockIdx.x >> 3);
    return b < count ? b : -1;
}

// a thread's node: plane pl of the workgroup, r = i + n*j in it
template <int N>
struct PlNode {
    int e, pl, r, i, j, k, node;
    bool active;
    __device__ __forceinline__ PlNode(int b, int tid)
    {
        using P = Pl<N>;
        e = b / P::groups;
        pl = tid / P::n2;
        r = tid - pl * P::n2;
        j = r / P::n;
        i = r - j * P::n;
        k = (b - e * P::groups) * P::planes + pl;
        active = pl < P::planes && k < P::n;
        node = r + P::n2 * k;
    }
};

// the four sides normal to the planes, in the order of the LDS arrays: xi-, xi+, eta-, eta+
__device__ __forceinline__ int plane_side(int s) { return s == 0 ? 5 : (s == 1 ? 3 : (s == 2 ? 2 : 4)); }

// side task t of a workgroup: position a (along j for the xi-, along i for the eta-sides) of side s in plane pl
template <int N>
struct PlSide {
    int pl, s, a, k, r;
    bool active;
    FaceTask f;
    __device__ __forceinline__ PlSide(int t, const PlNode<N>& nd, const Mesh& mesh)
    {
        using P = Pl<N>;
        constexpr int n = P::n;
        pl = t / (4 * n);
        s = (t - pl * 4 * n) / n;
        a = t - (pl * 4 + s) * n;
        k = nd.k - nd.pl + pl;
        active = pl < P::planes && k < n;
        r = s == 0 ? n * a : (s == 1 ? N + n * a : (s == 2 ? a : a + n * N));
        if (active) f = face_task<N>(nd.e, (plane_side(s) - 1) * P::n2 + a + n * k, mesh);
    }
    __device__ __forceinline__ int at(int c, int nc) const { return ((pl * 4 + s) * nc + c) * Pl<N>::n + a; }
};

// 0.5*SurfElem*(-L_master + L_slave) of the four lifted variables of a face node, from the neighbour's record and the
// own values (scale * s[qi[q] * n2], plane stride n2), and the side's normal
template <int N, typename T, typename TT>
__device__ __forceinline__ void plane_lift_flux(const FaceTask& f, const Mesh& mesh, const TT* __restrict__ utr,
                                                const T* s, const int* qi, T scale, const Gas<T>& gas, T* lf, T* nv)
{
    LiftOperands<T> p;
    load_lift_operands<N, T, TT>(f, mesh, utr, p);
    T uc[5], pr[6];
    trace_state(p.tr, gas, uc, pr);
    const T nb[4] = {pr[1], pr[2], pr[3], pr[5]};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const T own = scale * s[qi[q] * Pl<N>::n2];
        lf[q] = T(0.5) * p.se * (f.flip ? own - nb[q] : nb[q] - own);
    }
#pragma unroll
    for (int c = 0; c < 3; c++) nv[c] = p.nv[c];
}

// the BR1 gradients g[12] (layout of gradient_combine) of the workgroup's nodes.
//   s_q : [planes][nq][n2], the caller's u, v, w, T of its planes at planes qi[4], scaled by 1/scale (synchronised)
//   s_s : [planes][4][7][n] receives the lifting fluxes and normals of the sides (synchronised on return)
//   gze : the derivative along k of (u,v,w,T), from the caller
//   en  : normal of the node's k-side (k = 0 or N), out
template <int N, typename T, typename TT, class MT>
__device__ __forceinline__ void plane_gradient(const PlNode<N>& nd, int tid, const Mesh& mesh,
                                               const TT* __restrict__ utr, const MT& M, const T* s_q, int nq,
                                               const int* qi, T scale, T* s_s, const Gas<T>& gas, T LHm, T LHp,
                                               const T* gm, const T* gze, T* g, T* en)
{
    using P = Pl<N>;
    constexpr int n = P::n, n2 = P::n2;
    static_assert(4 * P::planes * n <= P::block, "one side task per thread");
    {
        const PlSide<N> sd(tid, nd, mesh);
        if (sd.active) {
            T lf[4], nv[3];
            plane_lift_flux<N, T, TT>(sd.f, mesh, utr, s_q + sd.pl * nq * n2 + sd.r, qi, scale, gas, lf, nv);
#pragma unroll
            for (int q = 0; q < 4; q++) s_s[sd.at(q, 7)] = lf[q];
#pragma unroll
            for (int c = 0; c < 3; c++) s_s[sd.at(4 + c, 7)] = nv[c];
        }
    }
    if (nd.active) {
        T gxi[4] = {0, 0, 0, 0}, get[4] = {0, 0, 0, 0};
        for (int l = 0; l <= N; l++) {
            const T di = M.dt(l, nd.i), dj = M.dt(l, nd.j);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const T* pq = s_q + (nd.pl * nq + qi[q]) * n2;
                gxi[q] = gxi[q] + di * pq[l + n * nd.j];
                get[q] = get[q] + dj * pq[nd.i + n * l];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const T a = scale * gxi[q], b = scale * get[q], c = gze[q];
            g[q] = gm[0] * a + gm[3] * b + gm[6] * c;
            g[4 + q] = gm[1] * a + gm[4] * b + gm[7] * c;
            g[8 + q] = gm[2] * a + gm[5] * b + gm[8] * c;
        }
        if (nd.k == 0 || nd.k == N) {
            const FaceTask f = face_task<N>(nd.e, (nd.k == 0 ? 0 : 5) * n2 + nd.r, mesh);
            T lf[4];
            plane_lift_flux<N, T, TT>(f, mesh, utr, s_q + nd.pl * nq * n2 + nd.r, qi, scale, gas, lf, en);
            const T LH = nd.k == 0 ? LHm : LHp;
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int c = 0; c < 3; c++) g[4 * c + q] = g[4 * c + q] + (lf[q] * en[c]) * LH;
        }
    }
    __syncthreads();
    if (nd.active) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const bool on = s == 0 ? nd.i == 0 : (s == 1 ? nd.i == N : (s == 2 ? nd.j == 0 : nd.j == N));
            if (!on) continue;
            const T* o = s_s + (nd.pl * 4 + s) * 7 * n + (s < 2 ? nd.j : nd.i);
            const T LH = (s & 1) ? LHp : LHm;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const T lf = o[q * n];
#pragma unroll
                for (int c = 0; c < 3; c++) g[4 * c + q] = g[4 * c + q] + (lf * o[(4 + c) * n]) * LH;
            }
        }
#pragma unroll
        for (int q = 0; q < 12; q++) g[q] = gm[9] * g[q];
    }
}

// F_v.n_master of one own face node (EvalNormalDiffFlux3D: -n.tau and -n.(tau.u + lambda grad T)) to its vtr slot
template <int N, typename T, typename TT>
__device__ __forceinline__ void plane_store_vtr(int e, int t, const Mesh& mesh, const Stress<T>& s, const T* nv,
                                                TT* __restrict__ vtr)
{
    constexpr int n2 = Pl<N>::n2;
    const FaceTask f = face_task<N>(e, t, mesh);
    TT* o = vtr + ((f.side * 2 + (f.flip ? 1 : 0)) * 4) * n2 + f.pq;
    o[0] = TT(-nv[0] * s.txx - nv[1] * s.txy - nv[2] * s.txz);
    o[n2] = TT(-nv[0] * s.txy - nv[1] * s.tyy - nv[2] * s.tyz);
    o[2 * n2] = TT(-nv[0] * s.txz - nv[1] * s.tyz - nv[2] * s.tzz);
    o[3 * n2] = TT(-nv[0] * s.qx - nv[1] * s.qy - nv[2] * s.qz);
}

// ---------------------------------------------------------------------------------------------------------
// k_vol_plane
// ---------------------------------------------------------------------------------------------------------
template <int N, typename T, typename TT, bool SPLIT>
__global__ void __launch_bounds__(Pl<N>::block, 4)
    k_vol_plane(int nElems, const double* __restrict__ U, Mesh mesh, const TT* __restrict__ utr, TT* __restrict__ vtr,
                const T* __restrict__ mats, GasD gd, T LHm, T LHp)
{
    using P = Pl<N>;
    constexpr int n = P::n, n2 = P::n2, n3 = P::n3, PL = P::planes;
    // split: halves of (rho,u,v,w,p,H,T); weak: u,v,w,T
    constexpr int nq = SPLIT ? 7 : 4, nf = SPLIT ? 4 : 5;
    __shared__ T s_q[PL * nq * n2];
    __shared__ T s_m[SPLIT ? PL * 3 * n2 : 1];  // halved metric of the current direction
    __shared__ T s_f[PL * (nf * n2 > 28 * n ? nf * n2 : 28 * n)];  // lifting fluxes of the sides, then the volume fluxes
    __shared__ Mats<N, T> M;
    const int b = plane_block(nElems * P::groups), tid = threadIdx.x;
    if (b < 0) return;
    const PlNode<N> nd(b, tid);
    const int e = nd.e, pl = nd.pl, r = nd.r;
    const T half = SPLIT ? T(0.5) : T(1);
    load_mats<N, T>(M, mats, tid, P::block);
    const Gas<T> gas = make_gas<T>(gd);
    T gm[10], uc[5], pr[6], H = T(0), hv[6];
    if (nd.active) {
        load_node_geo<N, T>(e, nd.node, mesh, gm);
        load_state<N, T>(e, nd.node, U, gd, uc, pr, H);
        T* q = s_q + pl * nq * n2 + r;
        if (SPLIT) {
#pragma unroll
            for (int c = 0; c < 5; c++) hv[c] = half * pr[c];
            hv[5] = half * H;
#pragma unroll
            for (int c = 0; c < 6; c++) q[c * n2] = hv[c];
            q[6 * n2] = half * pr[5];
        } else {
            q[0] = pr[1];
            q[n2] = pr[2];
            q[2 * n2] = pr[3];
            q[3 * n2] = pr[5];
        }
    }
    __syncthreads();
    // along k: the node's column from memory, for the derivative and the split pairs.  The diagonal pairs, which k_rhs
    // leaves out, stay in on all lines, as VolInt_splitForm_Kernel has them: DVolSurf(a,a), zero up to rounding, is the
    // residue that makes the rounded derivative matrix exact on constants (without it the N = 11 step is twice as far from
    // the FP64 result).
    T gze[4] = {0, 0, 0, 0}, tmp[5] = {0, 0, 0, 0, 0};
    if (nd.active) {
        const T* gk = GeoOf<T>::geo(mesh) + (long)e * 10 * n3 + 6 * n3 + r;
        const T hm[3] = {T(0.5) * gm[6], T(0.5) * gm[7], T(0.5) * gm[8]};
#pragma unroll 2
        for (int l = 0; l <= N; l++) {
            T c5[5], p6[6], Hl;
            load_state<N, T>(e, r + n2 * l, U, gd, c5, p6, Hl);
            const T d = M.dt(l, nd.k);
            gze[0] = gze[0] + d * p6[1];
            gze[1] = gze[1] + d * p6[2];
            gze[2] = gze[2] + d * p6[3];
            gze[3] = gze[3] + d * p6[5];
            if (SPLIT) {
                const T Mo[3] = {T(0.5) * gk[n2 * l], T(0.5) * gk[n3 + n2 * l], T(0.5) * gk[2 * n3 + n2 * l]};
                T G[5];
                split_volume_flux_pi_half<T>(hv[0], hv[1], hv[2], hv[3], hv[4], hv[5], half * p6[0], half * p6[1],
                                             half * p6[2], half * p6[3], half * p6[4], half * Hl, hm, Mo, G);
                const T dv = M.dvs(l, nd.k);
#pragma unroll
                for (int v = 0; v < 5; v++) tmp[v] = tmp[v] + dv * G[v];
            }
        }
    }
    Stress<T> st;
    {
        T g[12], en[3] = {0, 0, 0};
        const int qi[4] = {SPLIT ? 1 : 0, SPLIT ? 2 : 1, SPLIT ? 3 : 2, SPLIT ? 6 : 3};
        plane_gradient<N, T, TT>(nd, tid, mesh, utr, M, s_q, nq, qi, SPLIT ? T(2) : T(1), s_f, gas, LHm, LHp, gm, gze,
                                 g, en);
        if (nd.active) {
            stress(pr, g, gas, st);
            if (nd.k == 0) plane_store_vtr<N, T, TT>(e, r, mesh, st, en, vtr);
            if (nd.k == N) plane_store_vtr<N, T, TT>(e, 5 * n2 + r, mesh, st, en, vtr);
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const bool on = s == 0 ? nd.i == 0 : (s == 1 ? nd.i == N : (s == 2 ? nd.j == 0 : nd.j == N));
                if (!on) continue;
                const int a = s < 2 ? nd.j : nd.i;
                const T* o = s_f + (pl * 4 + s) * 7 * n + a;
                const T nv[3] = {o[4 * n], o[5 * n], o[6 * n]};
                plane_store_vtr<N, T, TT>(e, (plane_side(s) - 1) * n2 + a + n * nd.k, mesh, st, nv, vtr);
            }
        }
    }
    __syncthreads();
    T ut[5] = {0, 0, 0, 0, 0};
#pragma unroll 1
    for (int d = 0; d < 2; d++) {
        T hm[3];
        if (nd.active) {
            T m[3], f[5];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                m[c] = d == 0 ? gm[c] : gm[3 + c];
                hm[c] = T(0.5) * m[c];
                if (SPLIT) s_m[(pl * 3 + c) * n2 + r] = hm[c];
            }
            transformed_flux<T, !SPLIT>(uc, pr, st, m, gas.hshift, f);
#pragma unroll
            for (int v = 0; v < nf; v++) s_f[(pl * nf + v) * n2 + r] = f[v + 5 - nf];
        }
        __syncthreads();
        if (nd.active) {
            const int idx = d == 0 ? nd.i : nd.j, s0 = d == 0 ? n * nd.j : nd.i, ss = d == 0 ? 1 : n;
            const T* pf = s_f + pl * nf * n2 + s0;
            for (int l = 0; l <= N; l++) {
                const T dh = M.dht(l, idx);
#pragma unroll
                for (int v = 0; v < nf; v++) ut[v + 5 - nf] = ut[v + 5 - nf] + dh * pf[v * n2 + ss * l];
            }
            if (SPLIT) {
                const T *pq = s_q + pl * nq * n2 + s0, *pm = s_m + pl * 3 * n2 + s0;
                for (int l = 0; l <= N; l++) {
                    const T *q = pq + ss * l, *m = pm + ss * l;
                    const T Mo[3] = {m[0], m[n2], m[2 * n2]};
                    T G[5];
                    split_volume_flux_pi_half<T>(hv[0], hv[1], hv[2], hv[3], hv[4], hv[5], q[0], q[n2], q[2 * n2],
                                                 q[3 * n2], q[4 * n2], q[5 * n2], hm, Mo, G);
                    const T dv = M.dvs(l, idx);
#pragma unroll
                    for (int v = 0; v < 5; v++) tmp[v] = tmp[v] + dv * G[v];
                }
            }
        }
        __syncthreads();
    }
    if (nd.active) {
        T f[5];
        transformed_flux<T, !SPLIT>(uc, pr, st, gm + 6, gas.hshift, f);
        T* o = static_cast<T*>(mesh.ws) + (long)e * P::ws + nd.node;
        if (SPLIT) {
#pragma unroll
            for (int v = 0; v < 5; v++) ut[v] = ut[v] + T(2) * tmp[v];
            if (sizeof(T) == 4) ut[4] = ut[4] + T(gd.href) * (T(2) * tmp[0]);  // the enthalpy offset, as in k_rhs
        }
#pragma unroll
        for (int v = 0; v < 5; v++) o[v * n3] = ut[v];
#pragma unroll
        for (int v = 5 - nf; v < 5; v++) o[(5 + v) * n3] = f[v];
    }
}

// ---------------------------------------------------------------------------------------------------------
// k_upd_plane: stages as k_rhs (st.mode 0: Ut; 1: LSERK register update in place or from U to Uout)
// ---------------------------------------------------------------------------------------------------------
// flux of face node t = (ls-1)*n2 + ab, whose volume node is `node`, signed for the own element
template <int N, typename T, typename TT, bool SPLIT, int RIEMANN>
__device__ __forceinline__ void plane_face_flux(int e, const FaceTask& f, int node, const double* U, const Mesh& mesh,
                                                const TT* __restrict__ utr, const TT* __restrict__ vtr,
                                                const GasD& gd, const Gas<T>& gas, T* F)
{
    constexpr int n2 = Pl<N>::n2, n3 = Pl<N>::n3;
    const long own = f.side * 2 + (f.flip ? 1 : 0), nb = f.side * 2 + (f.flip ? 0 : 1);
    T Uo[5], Un[5], fv[8];
    {
        const double* uo = U + (long)e * 5 * n3 + node;
        double c[5], tr[5];
#pragma unroll
        for (int v = 0; v < 5; v++) c[v] = uo[v * n3];
        trace_record<sizeof(TT) == 4>(c, gd.kappa, gd.pref, tr);
#pragma unroll
        for (int v = 0; v < 5; v++) Uo[v] = T(TT(tr[v]));
    }
#pragma unroll
    for (int v = 0; v < 5; v++) Un[v] = T(utr[(nb * 5 + v) * n2 + f.pq]);
    face_flux<N, T, TT, SPLIT, RIEMANN, true>(Uo, Un, fv, vtr + own * 4 * n2 + f.pq, vtr + nb * 4 * n2 + f.pq,
                                              GeoOf<T>::fgeo(mesh) + f.side * 10 * n2 + f.pq, n2, f.flip, gas, F);
    const T sg = f.flip ? T(-1) : T(1);
#pragma unroll
    for (int v = 0; v < 5; v++) F[v] = sg * F[v];
}

template <int N, typename T, typename TT, bool SPLIT, int RIEMANN>
__global__ void __launch_bounds__(Pl<N>::block, 4)
    k_upd_plane(int nElems, const double* U, double* Uout, Mesh mesh, const TT* __restrict__ utr,
                const TT* __restrict__ vtr, TT* __restrict__ utr_next, double* __restrict__ Ut,
                double* __restrict__ Kreg, const T* __restrict__ mats, GasD gd, T LHm, T LHp, Stage st)
{
    using P = Pl<N>;
    constexpr int n = P::n, n2 = P::n2, n3 = P::n3, PL = P::planes;
    constexpr int nf = SPLIT ? 4 : 5;
    __shared__ T s_res[PL * 4 * 5 * n];
    const int b = plane_block(nElems * P::groups), tid = threadIdx.x;
    if (b < 0) return;
    const PlNode<N> nd(b, tid);
    const int e = nd.e, r = nd.r;
    const Gas<T> gas = make_gas<T>(gd);
    {
        const PlSide<N> sd(tid, nd, mesh);
        if (sd.active) {
            T F[5];
            plane_face_flux<N, T, TT, SPLIT, RIEMANN>(e, sd.f, sd.r + n2 * sd.k, U, mesh, utr, vtr, gd, gas, F);
#pragma unroll
            for (int v = 0; v < 5; v++) s_res[sd.at(v, 5)] = F[v];
        }
    }
    T ut[5] = {0, 0, 0, 0, 0};
    const bool kend = nd.active && (nd.k == 0 || nd.k == N);
    FaceTask fk;
    if (kend) {
        fk = face_task<N>(e, (nd.k == 0 ? 0 : 5) * n2 + r, mesh);
        T F[5];
        plane_face_flux<N, T, TT, SPLIT, RIEMANN>(e, fk, nd.node, U, mesh, utr, vtr, gd, gas, F);
        const T LH = nd.k == 0 ? LHm : LHp;
#pragma unroll
        for (int v = 0; v < 5; v++) ut[v] = F[v] * LH;
    }
    if (nd.active) {
        const T* w = static_cast<const T*>(mesh.ws) + (long)e * P::ws;
        const T* dh = mats + n2 + n * nd.k;  // D_Hat_T(l,k)
#pragma unroll
        for (int v = 0; v < 5; v++) ut[v] = ut[v] + w[v * n3 + nd.node];
#pragma unroll
        for (int l = 0; l <= N; l++) {
            const T d = dh[l];
#pragma unroll
            for (int v = 5 - nf; v < 5; v++) ut[v] = ut[v] + d * w[(5 + v) * n3 + r + n2 * l];
        }
    }
    __syncthreads();
    if (!nd.active) return;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const bool on = s == 0 ? nd.i == 0 : (s == 1 ? nd.i == N : (s == 2 ? nd.j == 0 : nd.j == N));
        if (!on) continue;
        const T* o = s_res + (nd.pl * 4 + s) * 5 * n + (s < 2 ? nd.j : nd.i);
        const T LH = (s & 1) ? LHp : LHm;
#pragma unroll
        for (int v = 0; v < 5; v++) ut[v] = ut[v] + o[v * n] * LH;
    }
    const double sJ = mesh.geo[((long)e * 10 + 9) * n3 + nd.node];
    const long at = (long)e * 5 * n3 + nd.node;
    if (st.mode == 0) {
#pragma unroll
        for (int v = 0; v < 5; v++) Ut[at + v * n3] = double(ut[v] * T(-1)) * sJ;
        return;
    }
    double unew[5], tr[5], kv[5];
#pragma unroll
    for (int v = 0; v < 5; v++) kv[v] = st.mRKA != 0.0 ? Kreg[at + v * n3] : 0.0;
    const double ak = source_into_register(st.src, (long)e * n3 + nd.node, st.mRKA, kv);
#pragma unroll
    for (int v = 0; v < 5; v++) {
        const double kk = kv[v] * ak + double(ut[v] * T(-1)) * sJ;
        if (!st.dropK) Kreg[at + v * n3] = kk;
        unew[v] = U[at + v * n3] + kk * st.bdt;
        Uout[at + v * n3] = unew[v];
    }
    // trace records of the new state, from the nodes on a face
    trace_record<sizeof(TT) == 4>(unew, gd.kappa, gd.pref, tr);
    auto put = [&](const FaceTask& f) {
        TT* o = utr_next + ((f.side * 2 + (f.flip ? 1 : 0)) * 5) * n2 + f.pq;
#pragma unroll
        for (int v = 0; v < 5; v++) o[v * n2] = TT(tr[v]);
    };
    if (kend) put(fk);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const bool on = s == 0 ? nd.i == 0 : (s == 1 ? nd.i == N : (s == 2 ? nd.j == 0 : nd.j == N));
        if (on) put(face_task<N>(e, (plane_side(s) - 1) * n2 + (s < 2 ? nd.j : nd.i) + n * nd.k, mesh));
    }
}

// ---------------------------------------------------------------------------------------------------------
// k_grad_plane: k_grad for these degrees (BR1 volume gradients of (u,v,w,T) for analysis, planes 0..11 of gvol
// [e][15][n3] in FP64)
// ---------------------------------------------------------------------------------------------------------
template <int N, typename T, typename TT>
__global__ void __launch_bounds__(Pl<N>::block)
    k_grad_plane(int nElems, const double* __restrict__ U, Mesh mesh, const TT* __restrict__ utr,
                 const T* __restrict__ mats, GasD gd, T LHm, T LHp, double* __restrict__ gvol)
{
    using P = Pl<N>;
    constexpr int n = P::n, n2 = P::n2, n3 = P::n3;
    __shared__ T s_q[P::planes * 4 * n2];
    __shared__ T s_s[P::planes * 28 * n];
    __shared__ MatsD<N, T> M;
    const int b = plane_block(nElems * P::groups), tid = threadIdx.x;
    if (b < 0) return;
    const PlNode<N> nd(b, tid);
    load_mats<N, T>(M, mats, tid, P::block);
    const Gas<T> gas = make_gas<T>(gd);
    T gm[10], uc[5], pr[6], H, gze[4] = {0, 0, 0, 0}, g[12], en[3];
    if (nd.active) {
        load_node_geo<N, T>(nd.e, nd.node, mesh, gm);
        load_state<N, T>(nd.e, nd.node, U, gd, uc, pr, H);
        T* q = s_q + nd.pl * 4 * n2 + nd.r;
        q[0] = pr[1];
        q[n2] = pr[2];
        q[2 * n2] = pr[3];
        q[3 * n2] = pr[5];
    }
    __syncthreads();
    if (nd.active)
        for (int l = 0; l <= N; l++) {
            load_state<N, T>(nd.e, nd.r + n2 * l, U, gd, uc, pr, H);
            const T d = M.dt(l, nd.k);
            gze[0] = gze[0] + d * pr[1];
            gze[1] = gze[1] + d * pr[2];
            gze[2] = gze[2] + d * pr[3];
            gze[3] = gze[3] + d * pr[5];
        }
    const int qi[4] = {0, 1, 2, 3};
    plane_gradient<N, T, TT>(nd, tid, mesh, utr, M, s_q, 4, qi, T(1), s_s, gas, LHm, LHp, gm, gze, g, en);
    if (nd.active) {
        double* o = gvol + (long)nd.e * 15 * n3 + nd.node;
#pragma unroll
        for (int q = 0; q < 12; q++) o[q * n3] = double(g[q]);
    }
}

}  // namespace galx
