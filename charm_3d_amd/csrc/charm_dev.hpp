// charm_dev.hpp -- the FP32 residual in deviation form (one species,
// constant gamma; LF, HLLC and central fluxes).
//
// Every chunk of the stage kernel picks a reference state U_r (the cell mean
// of its first leaf, taken as FP32 primitive values rho_r, u_r, p_r; its
// conserved values follow exactly in FP64).  All fluxes of the chunk's faces
// and volume points are evaluated as F(U) - F(U_r), with every term written
// so that no two O(|F|) quantities are subtracted: velocity deviations
// du = (dm - u_r drho) / rho, kinetic-energy deviation dK = (dm . u + rho_r
// u_r . du) / 2, dp = (gamma - 1)(dE - dK), and for HLLC the contact-speed
// offsets S* - u_K = (dp_R - dp_L - a_{R|L} (du_R - du_L)) / (a_L - a_R) with
// a_K = rho_K (S_K - u_K).  The dropped constant flux F(U_r) has an exactly
// zero DG residual (divergence theorem with the exact quadrature of the
// linear basis: sum over faces of F_r . n phi_k minus the volume integral of
// F_r . grad phi_k vanishes for every k, hanging faces included), so the
// residual of F - F(U_r) is the residual of F.  The FP32 rounding is then
// relative to the deviations (about 1% of |F| on the benchmark's perturbed
// Riemann box) instead of to |F| itself.
//
// The algebra is the reference's (src/charm_fluxes.c:255-315 LF, 319-437 HLLC
// x-split core, 513-559 central; src/models/euler/charm_model.c:66-132 volume
// fluxes); the FP64 path keeps the reference's arithmetic.
#pragma once
#include <hip/hip_runtime.h>
#include "charm_device.hpp"

namespace charm {

// chunk reference state: FP32 definitions and the FP64 conserved values they
// imply (m_r = rho_r u_r, E_r = p_r / (gamma - 1) + rho_r |u_r|^2 / 2)
struct DevRef {
    float r, u[3], p;
    float m[3], E, Epp;          // rounded rho_r u_r, E_r, E_r + p_r (multiply small terms only)
    double c0[5];                // exact (m_r[3], E_r, rho_r): subtracted from coefficient 0
    float c0h[5], c0l[5];        // c0 as the sum of two floats, c0h = c0 rounded
    float gam, gm1, gq;          // gamma, gamma - 1, (gamma + 1) / (2 gamma)
};

// reference from a cell mean (ru, rv, rw, re, rho), any finite positive
// density; a non-physical mean gives another (still exact) definition
__device__ __forceinline__ DevRef make_ref(const DevParams &P, double m0, double m1, double m2, double e0, double r0)
{
    DevRef R;
    R.gam = P.gam_f;
    R.gm1 = R.gam - 1.f;
    R.gq = (R.gam + 1.f) / (2.f * R.gam);
    if (!(r0 > 0.0) || !(r0 < 1e300)) { r0 = 1.0; m0 = m1 = m2 = 0.0; e0 = 1.0; }
    R.r = (float) r0;
    const double ri = 1.0 / (double) R.r;
    R.u[0] = (float) (m0 * ri); R.u[1] = (float) (m1 * ri); R.u[2] = (float) (m2 * ri);
    double kr = 0.0;
    #pragma unroll
    for (int d = 0; d < 3; d++) {
        R.c0[d] = (double) R.r * (double) R.u[d];          // exact product of two floats
        kr += R.c0[d] * (double) R.u[d];
    }
    kr *= 0.5;
    R.p = (float) ((double) R.gm1 * (e0 - kr));
    R.c0[3] = (double) R.p / (double) R.gm1 + kr;
    R.c0[4] = (double) R.r;
    #pragma unroll
    for (int d = 0; d < 3; d++) R.m[d] = (float) R.c0[d];
    #pragma unroll
    for (int i = 0; i < 5; i++) {
        R.c0h[i] = (float) R.c0[i];
        R.c0l[i] = (float) (R.c0[i] - (double) R.c0h[i]);
    }
    R.E = (float) R.c0[3];
    R.Epp = (float) (R.c0[3] + (double) R.p);
    return R;
}

// v_a of (v0, v1, v2) for a runtime axis a.  The arguments are values: a
// conditional over the lvalues R.u[0], R.u[1] would select their address,
// which keeps the whole reference record in private memory.
template <typename T>
__device__ __forceinline__ T vpick3(int a, T v0, T v1, T v2)
{
    return a == 0 ? v0 : (a == 1 ? v1 : v2);
}

// the reference with its velocity and momentum in the frame (a, t1, t2) of a
// boundary face normal to axis a (t1 the lower other axis)
__device__ __forceinline__ DevRef frame_ref(const DevRef &R, int a)
{
    DevRef Q = R;
    Q.u[0] = vpick3(a, R.u[0], R.u[1], R.u[2]);
    Q.u[1] = vpick3(a, R.u[1], R.u[0], R.u[0]);
    Q.u[2] = vpick3(a, R.u[2], R.u[2], R.u[1]);
    Q.m[0] = vpick3(a, R.m[0], R.m[1], R.m[2]);
    Q.m[1] = vpick3(a, R.m[1], R.m[0], R.m[0]);
    Q.m[2] = vpick3(a, R.m[2], R.m[2], R.m[1]);
    return Q;
}

// element coefficients as deviations: coefficient 0 minus the reference,
// slopes as they are.  An FP64 state subtracts in FP64 (one rounding of the
// difference); an FP32 state subtracts the two-float reference c0h + c0l in
// FP32, (x - c0h) - c0l, two roundings, each relative to the deviation.
template <typename S>
__device__ __forceinline__ void load_dev(const S *__restrict__ U, int64_t n, int e, const DevRef &R, float *u)
{
    #pragma unroll
    for (int i = 0; i < 20; i++) {
        const S x = ldp<S>(U, n, i, e);
        if constexpr (sizeof(S) == 4)
            u[i] = (i & 3) ? x : (x - R.c0h[i >> 2]) - R.c0l[i >> 2];
        else
            u[i] = (i & 3) ? (float) x : (float) ((double) x - R.c0[i >> 2]);
    }
}

// The pointwise functions below spell out their fused multiply-adds and let
// the compiler form no others, so that the result of a point from its traces
// does not depend on the kernel it is inlined into.  (The traces at volume
// points, the sums over points and faces and the update are the compiler's.)

// state at a point from its deviation trace t = (dm[3], dE, drho); x = dE less
// the kinetic-energy deviation, dp = (gamma - 1) x
struct DPrim {
    float r, ri, u[3], p, E, cz;
    float dr, dm[3], du[3], dE, dp, x;
};

__device__ __forceinline__ void dev_prim(const DevRef &R, const float *t, DPrim &q)
{
    #pragma clang fp contract(off)
    q.dm[0] = t[0]; q.dm[1] = t[1]; q.dm[2] = t[2]; q.dE = t[3]; q.dr = t[4];
    q.r = R.r + q.dr;
    q.ri = rcp(q.r);
    #pragma unroll
    for (int d = 0; d < 3; d++) {
        const float w = fmaf(-q.dr, R.u[d], q.dm[d]);
        q.du[d] = w * q.ri;
        q.u[d] = fmaf(q.ri, w, R.u[d]);
    }
    float k = q.dm[1] * q.u[1];
    k = fmaf(q.dm[0], q.u[0], k);
    k = fmaf(q.dm[2], q.u[2], k);
    #pragma unroll
    for (int d = 0; d < 3; d++) k = fmaf(q.du[d], R.m[d], k);
    q.x = fmaf(-0.5f, k, q.dE);
    q.dp = R.gm1 * q.x;
    q.p = fmaf(R.gm1, q.x, R.p);
    q.E = R.E + q.dE;
    q.cz = dsqrt(q.ri * (R.gam * q.p));
}

// deviation state of a full primitive state (exterior states of boundary
// faces other than the transmissive one): plain FP32 accuracy
__device__ __forceinline__ void dev_from_prim(const DevRef &R, const Prim<float, 1> &p, DPrim &q)
{
    q.r = p.r; q.ri = rcp(p.r);
    const float v[3] = {p.u, p.v, p.w};
    #pragma unroll
    for (int d = 0; d < 3; d++) {
        q.u[d] = v[d];
        q.du[d] = v[d] - R.u[d];
        q.dm[d] = p.r * v[d] - R.m[d];
    }
    q.p = p.p; q.dp = p.p - R.p;
    q.E = p.r * p.e_tot; q.dE = q.E - R.E;
    q.dr = p.r - R.r;
    q.cz = p.cz;
}

// full primitive state of a deviation state (input of the BC functions)
__device__ __forceinline__ void prim_of_dev(const DevParams &P, const DevRef &R, const DPrim &q, Prim<float, 1> &p)
{
    p.r = q.r; p.u = q.u[0]; p.v = q.u[1]; p.w = q.u[2];
    p.p = q.p; p.cz = q.cz; p.gam = R.gam;
    p.e_tot = q.E * q.ri;
    p.e = q.p * q.ri * rcp(R.gm1);
    p.cv = P.cv_f;
    p.m = P.m_f;
    p.c[0] = 1.f;
}

// Fluxes of two point states across a face normal to axis ax, minus F(U_r);
// q in the states' component order.  The axis may differ between lanes: the
// normal components are picked by selects, so that one code path serves the
// three axes with the components' sums in one order.  (On an interior face
// dp_R - dp_L is one fused step from the states' x.)

// HLLC (src/charm_fluxes.c:319-437): the upwind branches are the physical flux
// deviation, the star branch adds S_K (U*_K - U_K) =
// S_K g (rho_K S_K, rho_K ut1, rho_K ut2, E_K + a_K S* + p_K, rho_K),
// g = (S* - u_K) / (S_K - S*)
template <bool BND>
__device__ __forceinline__ bool hllc_dev(const DPrim &L, const DPrim &Rt, const DevRef &rf, int ax, float *q)
{
    #pragma clang fp contract(off)
    const float unl = vpick3(ax, L.u[0], L.u[1], L.u[2]), unr = vpick3(ax, Rt.u[0], Rt.u[1], Rt.u[2]);
    const float dnl = vpick3(ax, L.du[0], L.du[1], L.du[2]), dnr = vpick3(ax, Rt.du[0], Rt.du[1], Rt.du[2]);
    const float pv = 0.5f * (unr - unl) * -0.25f * (L.r + Rt.r) * (L.cz + Rt.cz);
    const float p_star = fmaxf(0.f, fmaf(0.5f, L.p + Rt.p, pv));
    // c_K q_K with q_K = sqrt(1 + gq (p* / p_K - 1)) for p* > p_K, else 1, as
    // one root: c_K q_K = sqrt(gamma / rho_K (p_K + gq max(p* - p_K, 0)))
    float sl = unl - dsqrt(rf.gam * L.ri * fmaf(rf.gq, fmaxf(0.f, p_star - L.p), L.p));
    float sr = unr + dsqrt(rf.gam * Rt.ri * fmaf(rf.gq, fmaxf(0.f, p_star - Rt.p), Rt.p));
    if (sl > sr) { const float t = sl; sl = sr; sr = t; }
    const float wl = sl - unl, wr = sr - unr, al = L.r * wl, ar = Rt.r * wr;
    const float dpn = BND ? Rt.dp - L.dp : fmaf(rf.gm1, Rt.x, -L.dp), dun = dnr - dnl;
    const float den = rcp(fmaf(L.r, wl, -ar));
    const float nl = fmaf(-dun, ar, dpn);
    float dl = nl * den;                            // S* - u_L
    float dr = fmaf(-dun, al, dpn) * den;           // S* - u_R
    float s_star = fmaf(nl, den, unl);
    if (s_star < sl) { s_star = sl; dl = wl; dr = sl - unr; }
    if (s_star > sr) { s_star = sr; dl = sr - unl; dr = wr; }
    const bool ok = (sl <= s_star) && (s_star <= sr);
    // one branch-free body: the upwind side of a supersonic face (sl >= 0:
    // left, sr <= 0: right) with no star term, else the star region of the
    // side s* falls on
    const bool sup = (sl >= 0.f) || (sr <= 0.f);
    const bool left = (sl >= 0.f) || (!(sr <= 0.f) && s_star >= 0.f);
    const float un = sel(left, unl, unr), dn = sel(left, dnl, dnr), r = sel(left, L.r, Rt.r), p = sel(left, L.p, Rt.p);
    const float E = sel(left, L.E, Rt.E), dE = sel(left, L.dE, Rt.dE), dp = sel(left, L.dp, Rt.dp);
    const float sk = left ? sl : sr, dk = left ? dl : dr;
    const float sg = sup ? 0.f : sk * dk * rcp(sk - s_star);          // S_K g
    float dm[3];
    #pragma unroll
    for (int j = 0; j < 3; j++) dm[j] = sel(left, L.dm[j], Rt.dm[j]);
    const float dmn = vpick3(ax, dm[0], dm[1], dm[2]);
    const float mn = vpick3(ax, rf.m[0], rf.m[1], rf.m[2]);
    const float qn = fmaf(r * sk, sg, fmaf(mn, dn, un * dmn) + dp);
    #pragma unroll
    for (int j = 0; j < 3; j++) {
        const float u = sel(left, L.u[j], Rt.u[j]);
        const float qt = fmaf(r * u, sg, fmaf(un, dm[j], dn * rf.m[j]));
        q[j] = ax == j ? qn : qt;
    }
    q[3] = fmaf(dn, rf.Epp, un * (dp + dE));
    q[3] = fmaf(sg, p + fmaf(s_star, r * (sk - un), E), q[3]);
    q[4] = fmaf(r, sg, dmn);
    return ok;
}

// Lax-Friedrichs / central (src/charm_fluxes.c:255-315, 513-559)
__device__ __forceinline__ void lf_dev(const DPrim &L, const DPrim &Rt, const DevRef &rf, int ax, float *q,
                                       bool central)
{
    #pragma clang fp contract(off)
    float f[2][5], un[2];
    #pragma unroll
    for (int s = 0; s < 2; s++) {
        const DPrim &K = s ? Rt : L;
        un[s] = vpick3(ax, K.u[0], K.u[1], K.u[2]);
        const float dn = vpick3(ax, K.du[0], K.du[1], K.du[2]);
        #pragma unroll
        for (int j = 0; j < 3; j++) f[s][j] = fmaf(K.dm[j], un[s], rf.m[j] * dn) + (ax == j ? K.dp : 0.f);
        f[s][3] = fmaf(rf.Epp, dn, un[s] * (K.dE + K.dp));
        f[s][4] = vpick3(ax, K.dm[0], K.dm[1], K.dm[2]);
    }
    const float alpha = central ? 0.f : fmaxf(fabsf(un[0]) + L.cz, fabsf(un[1]) + Rt.cz);
    #pragma unroll
    for (int j = 0; j < 3; j++) q[j] = 0.5f * fmaf(-alpha, Rt.dm[j] - L.dm[j], f[1][j] + f[0][j]);
    q[3] = 0.5f * fmaf(-alpha, Rt.dE - L.dE, f[1][3] + f[0][3]);
    q[4] = 0.5f * fmaf(-alpha, Rt.dr - L.dr, f[1][4] + f[0][4]);
}

// flux deviations along the three axes at a volume point
__device__ __forceinline__ void phys_dev(const DPrim &q, const DevRef &rf, float (*F)[5])
{
    #pragma clang fp contract(off)
    const float h = fmaf(rf.gm1, q.x, q.dE);               // dE + dp
    #pragma unroll
    for (int d = 0; d < 3; d++) {
        #pragma unroll
        for (int j = 0; j < 3; j++) {
            F[d][j] = fmaf(q.du[j], rf.m[d], q.dm[d] * q.u[j]);
            if (d == j) F[d][j] = fmaf(rf.gm1, q.x, F[d][j]);
        }
        F[d][3] = fmaf(q.du[d], rf.Epp, q.u[d] * h);
        F[d][4] = q.dm[d];
    }
}

template <int FLUX, bool BND>
__device__ __forceinline__ bool flux_dev(const DPrim &L, const DPrim &Rt, const DevRef &rf, int ax, float *q)
{
    if constexpr (FLUX == FLUX_HLLC) {
        return hllc_dev<BND>(L, Rt, rf, ax, q);
    } else {
        lf_dev(L, Rt, rf, ax, q, FLUX == FLUX_CD);
        return true;
    }
}

// whether a stage kernel instance evaluates its FP32 residual in deviation form
template <typename R, int NC, int FLUX, int PH>
constexpr bool uses_dev()
{
    return sizeof(R) == 4 && NC == 1 && PH == 0 && FLUX != FLUX_GODUNOV;
}

} // namespace charm
