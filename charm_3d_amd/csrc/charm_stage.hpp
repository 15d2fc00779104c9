// charm_stage.hpp -- the stage kernel of the DG residual / time-step path
// (included by the translation units that instantiate it per precision and
// physics variant, so that they compile in parallel).
//
// State layout (structure of arrays): U[(4 v + k) n + e] for element e of n,
// variable v = ru rv rw re rc[..], Taylor coefficient k (1, (x-xc)/h,
// (y-yc)/h, (z-zc)/h): a wave's per-element accesses are unit-stride.
//
// One RK stage = k_stage over workgroup chunks (at most one element per
// thread of the 128- or 256-thread workgroup, Morton-consecutive, and a cap
// on the chunk's faces that sizes its LDS):
//   phase 1  one thread per (sub)face touching the chunk: both traces at the
//            six face Gauss points, the Riemann flux, and the three flux
//            moments per variable (sum q wJ, sum q phi_t1 wJ, sum q phi_t2 wJ in
//            the small side's face frame) written to LDS;
//   phase 2  one thread per element: volume integral at the 8 Gauss points,
//            gather of its face moments from LDS (no atomics: a fixed slot
//            list per element), A^-1 (diagonal on the cube octree) and the
//            SSP-RK update / combine, one write of the new state.
// Faces shared by two chunks are evaluated by both (each keeps its side).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "charm_device.hpp"
#include "charm_dev.hpp"
#include "charm_kernels.h"

namespace charm {

// SSP-RK combines rk_1 (c = c/4 + 3 c_old/4) and rk_2 (c = 2c/3 + c_old/3)
// in the reference's operation order, src/models/ns/charm_model.c:136-184
template <typename R>
__device__ __forceinline__ R rk_combine(int mode, R w, R u0)
{
    if (mode == 1) { R c = w * R(0.25); return c + R(0.75) * u0; }
    R c = w * R(2);
    c /= R(3);
    return c + u0 / R(3);
}

// per-(v, k) array bases are wave-uniform (scalar registers); the element
// index is the 32-bit per-lane offset
template <typename R, int NV>
__device__ __forceinline__ void load_elem(const R *__restrict__ U, int64_t n, int e, R *u)
{
    #pragma unroll
    for (int i = 0; i < 4 * NV; i++) u[i] = ldp<R>(U, n, i, e);
}

// load a state stored in S into the arithmetic type R
template <typename S, typename R, int NV>
__device__ __forceinline__ void load_conv(const S *__restrict__ U, int64_t n, int e, R *u)
{
    #pragma unroll
    for (int i = 0; i < 4 * NV; i++) u[i] = (R) ldp<S>(U, n, i, e);
}

template <typename R, int NV>
__device__ __forceinline__ void trace(const R *u, R px, R py, R pz, R *t)
{
    #pragma unroll
    for (int v = 0; v < NV; v++)
        t[v] = u[4*v] + px * u[4*v+1] + py * u[4*v+2] + pz * u[4*v+3];
}

// spread (normal, t1, t2) components onto (x, y, z)
template <typename R>
__device__ __forceinline__ void to_xyz(int a, R n, R t1, R t2, R &x, R &y, R &z)
{
    x = (a == 0) ? n : t1;
    y = (a == 1) ? n : ((a == 0) ? t1 : t2);
    z = (a == 2) ? n : t2;
}

// Element coefficients for a face normal to axis ax: the slopes in the face's
// order (n, t1 < t2), so that one code path serves the faces of all three
// axes and a wave that straddles two orientations does not run the face code
// twice (with the axis as a template argument 0.84 of the lanes were active at
// level 7 in FP32, 0.65 at level 6 in FP64).  The kernel is bound by VALU
// issue: 458 -> 422 us at 2,097,152 leaves in FP32, 152 -> 141 us at 262,144
// in FP64.  The planes are picked by the lane's byte offset.  The momentum components keep their order in the
// deviation form (DEV; deviations from the reference, as load_dev), whose
// flux picks the normal ones; else they follow into the frame by selects.
template <typename R>
__device__ __forceinline__ void frame_momentum(int ax, R *u)
{
    #pragma unroll
    for (int k = 0; k < 4; k++) {
        const R x = u[k], y = u[4 + k], z = u[8 + k];
        u[k] = vpick3(ax, x, y, z);
        u[4 + k] = ax == 0 ? y : x;
        u[8 + k] = ax == 2 ? y : z;
    }
}

template <typename S, typename R, int NC, bool DEV>
__device__ __forceinline__ void load_frame(const S *__restrict__ U, int64_t n, int e, int ax, const DevRef &rf, R *u)
{
    constexpr int NV = 4 + NC;
    const int np = (int) (n * (int64_t) sizeof(S)), o0 = e * (int) sizeof(S);
    const int off[4] = {o0, o0 + (ax == 0 ? np : (ax == 1 ? 2 * np : 3 * np)), o0 + (ax == 0 ? 2 * np : np),
                        o0 + (ax == 2 ? 2 * np : 3 * np)};
    #pragma unroll
    for (int v = 0; v < NV; v++)
        #pragma unroll
        for (int k = 0; k < 4; k++) {
            const S x = ldo<S>(U, n, v, off[k]);
            if constexpr (DEV && sizeof(S) == 4) u[4 * v + k] = k ? x : (x - rf.c0h[v]) - rf.c0l[v];
            else if constexpr (DEV) u[4 * v + k] = k ? (float) x : (float) ((double) x - rf.c0[v]);
            else u[4 * v + k] = (R) x;
        }
    if constexpr (!DEV) frame_momentum<R>(ax, u);
}

// The points of a face in its two sides' coordinates: scale and tangential
// offsets.  The big side of a hanging face sees the small face's points at
// delta + offset / 2 in its own units.
template <typename R>
struct FaceMap {
    R m0, o01, o02, m1, o11, o12;
    __device__ __forceinline__ FaceMap(int kind, int sub)
    {
        const R d1 = (sub & 1) ? R(0.25) : R(-0.25), d2 = (sub & 2) ? R(0.25) : R(-0.25);
        const bool big0 = kind == FACE_HANG1, big1 = kind == FACE_HANG0;
        m0 = big0 ? R(0.5) : R(1); m1 = big1 ? R(0.5) : R(1);
        o01 = big0 ? d1 : R(0); o02 = big0 ? d2 : R(0);
        o11 = big1 ? d1 : R(0); o12 = big1 ? d2 : R(0);
    }
};

// the value on the face (its normal-direction part is the same at all points)
// takes coefficient 0's place
template <typename R, int NV>
__device__ __forceinline__ void to_face(R pn, R *u)
{
    #pragma unroll
    for (int v = 0; v < NV; v++) u[4*v] = fma(pn, u[4*v+1], u[4*v]);
}

template <typename R, int NV>
__device__ __forceinline__ void face_trace(const R *u, R q1, R q2, R *t)
{
    #pragma unroll
    for (int v = 0; v < NV; v++) t[v] = fma(q2, u[4*v+3], fma(q1, u[4*v+2], u[4*v]));
}

// The flux q at the face point of offsets g1, g2 from the two sides (to_face;
// u1 unused on a boundary face, whose state and normal are mirrored so that
// the outward normal is +n), in the frame; DEV: q is F - F(U_r) (charm_dev.hpp),
// in the frame on a boundary face, in global order (normal axis ax) on others.
// dir0, s: the boundary face's direction and outward sign along its axis.
// tl / tr (PH = 1, may be null): each side's EOS closure at this point from
// the point pass, its planes kMemoRows * ts apart
template <typename R, int NC, int FLUX, bool BND, int PH, bool DEV>
__device__ __forceinline__ bool point_flux(const DevParams &P, const R *u0, const R *u1, const FaceMap<R> &fm, R g1, R g2, int dir0, R s,
                                           const DevRef &rf, const R *tl, const R *tr, int64_t ts, R *q)
{
    constexpr int NV = 4 + NC;
    R t[NV];
    face_trace<R, NV>(u0, BND ? g1 : fma(fm.m0, g1, fm.o01), BND ? g2 : fma(fm.m0, g2, fm.o02), t);
    if constexpr (DEV) {
        DPrim dl, dr;
        dev_prim(rf, t, dl);
        if (BND) {
            if (P.bnd_type[dir0] == BND_OUTLET) {
                dr = dl;                   // transmissive: the exterior state is the interior one
            } else {
                Prim<float, 1> pl, pr;
                prim_of_dev(P, rf, dl, pl);
                pl.u *= s;
                bnd_state<float, 1, 0>(P, dir0, 0, s, pl, pr, dir0 >> 1);
                pr.u *= s;
                dev_from_prim(rf, pr, dr);
            }
        } else {
            face_trace<R, NV>(u1, fma(fm.m1, g1, fm.o11), fma(fm.m1, g2, fm.o12), t);
            dev_prim(rf, t, dr);
        }
        return flux_dev<FLUX, BND>(dl, dr, rf, BND ? 0 : dir0 >> 1, q);
    } else {
        Prim<R, NC> pl, pr;
        cons_to_prim<R, NC, PH>(P, t, pl, tl, kMemoRows * ts);
        if (BND) {
            pl.u *= s;
            bnd_state<R, NC, PH>(P, dir0, 0, s, pl, pr, dir0 >> 1);
            pl.u *= s;
            pr.u *= s;
        } else {
            face_trace<R, NV>(u1, fma(fm.m1, g1, fm.o11), fma(fm.m1, g2, fm.o12), t);
            cons_to_prim<R, NC, PH>(P, t, pr, tr, kMemoRows * ts);
        }
        return flux_x<R, NC, FLUX>(frame_state(pl), frame_state(pr), q);
    }
}

// Moments of one face from its two element states in the face's frame
// (load_frame): out[3][NV] = wJ * (sum q, sum q phi_t1, sum q phi_t2) over the
// six points, q and phi in the frame, phi_t the tangential Taylor coordinates
// of the small (or side-0) face.  tl / tr as point_flux's for point k at
// tl[k * ts] (global memory: the point loop is not unrolled, so a local array
// would sit in scratch).
template <typename R, int NC, int FLUX, bool BND, int PH, bool DEV>
__device__ __forceinline__ bool face_core(const DevParams &P, R *u0, R *u1, int kind, int sub, int dir0, R s,
                                          int lown, R *out, const DevRef &rf, const R *tl = nullptr,
                                          const R *tr = nullptr, int64_t ts = 0)
{
    constexpr int NV = 4 + NC;
    const R h = ldexp(R(1), -lown);
    const R wj = h * h * R(1.0 / 6.0);
    R S0[NV], S1[NV], S2[NV];
    #pragma unroll
    for (int v = 0; v < NV; v++) { S0[v] = R(0); S1[v] = R(0); S2[v] = R(0); }
    to_face<R, NV>(R(0.5), u0);
    if (!BND) to_face<R, NV>(R(-0.5), u1);
    const FaceMap<R> fm(kind, sub);
    bool ok = true;
    // a rolled loop over the points (k is wave-uniform: the point's constants
    // are scalar selects): a fifth of the unrolled code and fewer registers
    #pragma unroll 1
    for (int k = 0; k < 6; k++) {
        const R g1 = gp_t1<R>(k), g2 = gp_t2<R>(k);
        R q[NV];
        ok &= point_flux<R, NC, FLUX, BND, PH, DEV>(P, u0, u1, fm, g1, g2, dir0, s, rf, tl ? tl + k * ts : nullptr,
                                                    tr ? tr + k * ts : nullptr, ts, q);
        #pragma unroll
        for (int v = 0; v < NV; v++) { S0[v] += q[v]; S1[v] = fma(q[v], g1, S1[v]); S2[v] = fma(q[v], g2, S2[v]); }
    }
    #pragma unroll
    for (int v = 0; v < NV; v++) {
        out[v] = S0[v] * wj;
        out[NV + v] = S1[v] * wj;
        out[2 * NV + v] = S2[v] * wj;
    }
    if (BND) {
        #pragma unroll
        for (int m = 0; m < 3; m++) out[m * NV] *= s;
    }
    return ok;
}

// a boundary face's state and reference in its frame, mirrored to the outward
// normal +n
template <typename R, int NV, bool DEV>
__device__ __forceinline__ void mirror_side(int ax, R s, R *u, DevRef &rf)
{
    if constexpr (DEV) {
        frame_momentum<R>(ax, u);
        rf = frame_ref(rf, ax);
    }
    #pragma unroll
    for (int v = 0; v < NV; v++) u[4*v+1] *= s;
    #pragma unroll
    for (int k = 0; k < 4; k++) u[k] *= s;
    if constexpr (DEV) { rf.u[0] *= s; rf.m[0] *= s; }
}

// PH = 1: each side's point EOS closures from the point pass, at the side's
// own (sub)face slot 4 d + j (point k at k * n), or null
template <typename R, int PH>
__device__ __forceinline__ void face_closures(const StageArgs &A, int4 rec, const R *&tl, const R *&tr)
{
    tl = tr = nullptr;
    if (PH == 1 && A.tpt) {
        const R *TP = reinterpret_cast<const R *>(A.tpt);
        const int64_t n = A.n_elem;
        const int dir0 = rec.z & 7, kind = (rec.z >> 3) & 3, sub = (rec.z >> 5) & 3;
        const int s0 = 4 * dir0 + (kind == FACE_HANG1 ? sub : 0);
        const int s1 = 4 * (dir0 ^ 1) + (kind == FACE_HANG0 ? sub : 0);
        tl = TP + (int64_t) 6 * s0 * n + rec.x;
        if (kind != FACE_BND) tr = TP + (int64_t) 6 * s1 * n + rec.y;
    }
}

// One face record of a chunk: its moments into dst[3][NV] (global momentum
// order)
template <typename S, typename R, int NC, int FLUX, int PH, bool DEV>
__device__ __forceinline__ bool face_record(const DevParams &P, const S *__restrict__ U, int64_t n, int4 rec,
                                            int lev0, const DevRef &rf, R *dst, const R *tl, const R *tr)
{
    constexpr int NV = 4 + NC;
    const int dir0 = rec.z & 7, kind = (rec.z >> 3) & 3, sub = (rec.z >> 5) & 3, ax = dir0 >> 1;
    R ua[4 * NV], o[3 * NV];
    load_frame<S, R, NC, DEV>(U, n, rec.x, ax, rf, ua);
    bool ok;
    if (kind == FACE_BND) {
        const R s = (dir0 & 1) ? R(1) : R(-1);
        DevRef rx = rf;
        mirror_side<R, NV, DEV>(ax, s, ua, rx);
        ok = face_core<R, NC, FLUX, true, PH, DEV>(P, ua, ua, kind, sub, dir0, s, lev0, o, rx, tl, nullptr, n);
    } else {
        // side 0 of an interior face is the leaf on the lower side: s = +1
        R ub[4 * NV];
        load_frame<S, R, NC, DEV>(U, n, rec.y, ax, rf, ub);
        ok = face_core<R, NC, FLUX, false, PH, DEV>(P, ua, ub, kind, sub, dir0, R(1),
                                                    kind == FACE_HANG1 ? lev0 + 1 : lev0, o, rf, tl, tr, n);
    }
    // the frame's momentum moments back to global order by the LDS address
    const bool fr = !DEV || kind == FACE_BND;
    const int g0 = fr ? ax : 0, g1 = fr ? (ax == 0 ? 1 : 0) : 1, g2 = fr ? (ax == 2 ? 1 : 2) : 2;
    #pragma unroll
    for (int m = 0; m < 3; m++) {
        dst[m * NV + g0] = o[m * NV];
        dst[m * NV + g1] = o[m * NV + 1];
        dst[m * NV + g2] = o[m * NV + 2];
        #pragma unroll
        for (int v = 3; v < NV; v++) dst[m * NV + v] = o[m * NV + v];
    }
    return ok;
}

// The volume integral, src/models/euler/charm_model.c:66-132: with the Taylor
// basis on a cube, grad phi_k = e_k / h and phi_k(gp) = +-1/(2 sqrt 3), so
// int[v][1+d] -= (wJ/h) sum_gp F_d,v and the gravity term adds
// -g_v sum_gp rho phi_k wJ.
// volume_terms: the fluxes F_d at one Gauss point (signs of g) and the density
// there.  DEV: u holds deviation coefficients and F is F - F(U_r), the
// momentum, energy and mass fluxes along each axis as in phys_dev; the gravity
// term takes the full density.
// tk (PH = 1, may be null): the point's EOS closure, its planes kMemoRows * ts
// apart
template <typename R, int NC, int PH, bool DEV>
__device__ __forceinline__ R volume_terms(const DevParams &P, const R *u, int g, const DevRef &rf, const R *tk,
                                          int64_t ts, R (*F)[4 + NC])
{
    constexpr int NV = 4 + NC;
    const R ph = R(0.28867513459481288225);           // 1/(2 sqrt 3)
    const R px = (g & 1) ? ph : -ph, py = (g & 2) ? ph : -ph, pz = (g & 4) ? ph : -ph;
    R t[NV];
    trace<R, NV>(u, px, py, pz, t);
    if constexpr (DEV) {
        DPrim q;
        dev_prim(rf, t, q);
        phys_dev(q, rf, F);
        return q.r;
    } else {
        Prim<R, NC> p;
        cons_to_prim<R, NC, PH>(P, t, p, tk, kMemoRows * ts);
        const R vel[3] = {p.u, p.v, p.w};
        #pragma unroll
        for (int d = 0; d < 3; d++) {
            F[d][0] = t[d] * p.u + (d == 0 ? p.p : R(0));
            F[d][1] = t[d] * p.v + (d == 1 ? p.p : R(0));
            F[d][2] = t[d] * p.w + (d == 2 ? p.p : R(0));
            F[d][3] = t[d] * p.e_tot + p.p * vel[d];
            #pragma unroll
            for (int i = 0; i < NC; i++) F[d][4 + i] = t[d] * p.c[i];
        }
        return p.r;
    }
}

// tv (PH = 1, may be null): the EOS closure at volume point g starts at
// tv[g * ts]
template <typename R, int NC, int PH, bool DEV>
__device__ __forceinline__ void volume_integral(const DevParams &P, const R *u, R h, const DevRef &rf, R *res,
                                                const R *tv = nullptr, int64_t ts = 0)
{
    constexpr int NV = 4 + NC;
    const R ph = R(0.28867513459481288225);
    const R wj = h * h * h * R(0.125), f = wj * rcp(h);
    R SF[3][NV];
    R G[4] = {R(0), R(0), R(0), R(0)};
    #pragma unroll
    for (int d = 0; d < 3; d++)
        #pragma unroll
        for (int v = 0; v < NV; v++) SF[d][v] = R(0);
    #pragma unroll
    for (int g = 0; g < 8; g++) {
        R F[3][NV];
        const R r = volume_terms<R, NC, PH, DEV>(P, u, g, rf, tv ? tv + g * ts : nullptr, ts, F);
        #pragma unroll
        for (int d = 0; d < 3; d++)
            #pragma unroll
            for (int v = 0; v < NV; v++) SF[d][v] += F[d][v];
        G[0] += r; G[1] += r * ((g & 1) ? ph : -ph); G[2] += r * ((g & 2) ? ph : -ph);
        G[3] += r * ((g & 4) ? ph : -ph);
    }
    #pragma unroll
    for (int v = 0; v < NV; v++) {
        res[4*v+0] = R(0);
        res[4*v+1] = -SF[0][v] * f;
        res[4*v+2] = -SF[1][v] * f;
        res[4*v+3] = -SF[2][v] * f;
    }
    #pragma unroll
    for (int v = 0; v < 3; v++) {
        const R gv = cst<R>(P.grav[v], P.grav_f[v]);
        #pragma unroll
        for (int k = 0; k < 4; k++) res[4*v+k] -= gv * G[k] * wj;
    }
}

// the moments (M0, M1, M2) of one variable of a face record added to its
// leaf's integrals res[4] of that variable, from the given side
template <typename R>
__device__ __forceinline__ void slot_add(int info, int side, R M0, R M1, R M2, R *res)
{
    const int dir0 = info & 7, kind = (info >> 3) & 3, sub = (info >> 5) & 3;
    const R sg = side ? R(-1) : R(1);
    const R pa = ((dir0 & 1) ^ side) ? R(0.5) : R(-0.5);
    const bool big = (kind == FACE_HANG0 && side == 1) || (kind == FACE_HANG1 && side == 0);
    const R mu = big ? R(0.5) : R(1);
    const R d1 = big ? ((sub & 1) ? R(0.25) : R(-0.25)) : R(0);
    const R d2 = big ? ((sub & 2) ? R(0.25) : R(-0.25)) : R(0);
    const R m0 = sg * M0, m1 = sg * M1, m2 = sg * M2;
    R cx, cy, cz;
    to_xyz<R>(dir0 >> 1, pa * m0, mu * m1 + d1 * m0, mu * m2 + d2 * m0, cx, cy, cz);
    res[0] += m0;
    res[1] += cx;
    res[2] += cy;
    res[3] += cz;
}

// S: storage type of the state; R: arithmetic type of the residual (S = R,
// or the mixed mode S = double, R = float: FP32 fluxes and integrals, FP64
// state, update and combine).  PH = 0: constant-cp Euler terms; PH = 1: any
// cp (FP64 Newton T) and the viscous integrals of the Navier-Stokes model
// added before A^-1.
// PH = 1 reads the constants from device memory (runtime-indexed power
// series and BC records), PH = 0 from the by-value kernel argument
template <int PH>
__device__ __forceinline__ const DevParams &stage_params(const StageArgs &A, const DevParams &Pv)
{
    if constexpr (PH == 1) return *A.prm;
    else return Pv;
}

// the deviation reference of chunk c: the cell mean of its reference leaf
template <typename S>
__device__ __forceinline__ DevRef chunk_ref(const StageArgs &A, const DevParams &P, int c)
{
    const S *__restrict__ U = reinterpret_cast<const S *>(A.U);
    const int64_t n = A.n_elem;
    const int r = A.ch_ref[c];
    return make_ref(P, (double) U[r], (double) (U + 4 * n)[r], (double) (U + 8 * n)[r], (double) (U + 12 * n)[r],
                    (double) (U + 16 * n)[r]);
}

// The FP32 deviation-form instances are held to at most 168 VGPRs (three
// waves per SIMD) so that a change of the code cannot drop them below the
// occupancy their LDS allows; with the rolled point loop they need 114, and
// four 40 KB workgroups share a CU.  The FP64 ones are held to two waves, but
// for the exact Riemann solver with several species, which takes 264-308
// registers and spills 10-75 of them under that bound: stage with 85-leaf chunks
// at 32,768 / 83,672 / 262,144 leaves with one and two waves, us, two species
// 133 318 818 and 198 330 677, three 145 333 873 and 212 379 895, four 143 350
// 897 and 226 423 1,020.  Two species run a two-wave instance beyond 100,000
// leaves (launch_stage_bs).
template <typename R, int NC, int FLUX, int PH>
constexpr int stage_min_waves()
{
    return uses_dev<R, NC, FLUX, PH>() ? 3
           : (sizeof(R) == 8 && PH == 0 && (FLUX != FLUX_GODUNOV || NC == 1) ? 2 : 1);
}

template <typename S, typename R, int NC, int FLUX, int BS, int PH, int WAVES = stage_min_waves<R, NC, FLUX, PH>()>
__global__ __launch_bounds__(BS, WAVES)
void k_stage(StageArgs A, DevParams Pv)
{
    const DevParams &P = stage_params<PH>(A, Pv);
    constexpr int NV = 4 + NC;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    R *mom = reinterpret_cast<R *>(smem_raw);                       // [maxf][3][NV]
    int *finfo = reinterpret_cast<int *>(smem_raw + (size_t) A.max_faces * 3 * NV * sizeof(R));
    const S *__restrict__ U = reinterpret_cast<const S *>(A.U);
    const int c = xcd_block(A.n_xcd);
    if (c >= A.n_chunks) return;                 // whole workgroup exits together
    const int fb = A.ch_fbeg[c], fe = A.ch_fbeg[c + 1];
    const int eb = A.ch_ebeg[c], ee = A.ch_ebeg[c + 1];
    const int64_t n = A.n_elem;
    // FP32, one species: deviation form against the chunk's reference, the
    // same for every face and leaf of the chunk
    constexpr bool DEV = uses_dev<R, NC, FLUX, PH>();
    DevRef rf{};
    if constexpr (DEV) rf = chunk_ref<S>(A, P, c);
    bool ok = true;
    for (int f = fb + (int) threadIdx.x; f < fe; f += BS) {
        const int4 rec = A.cf4[f];
        R *dst = mom + (size_t) (f - fb) * 3 * NV;
        const int lev0 = A.level[rec.x];
        const R *pl, *pr;
        face_closures<R, PH>(A, rec, pl, pr);
        ok &= face_record<S, R, NC, FLUX, PH, DEV>(P, U, n, rec, lev0, rf, dst, pl, pr);
        finfo[f - fb] = rec.z;
    }
    __syncthreads();
    const int e = eb + (int) threadIdx.x;
    if (e < ee) {
        R u[4 * NV], res[4 * NV];
        const int lev = A.level[e];
        const R h = ldexp(R(1), -lev);
        // a leaf has at least six slots: their loads are in flight during the
        // volume integral (one dependent load per slot before)
        const int s_beg = A.slot_ptr[e], s_end = A.slot_ptr[e + 1];
        int sl6[6];
        #pragma unroll
        for (int k = 0; k < 6; k++) sl6[k] = A.slots[s_beg + k];
        if constexpr (DEV) load_dev<S>(U, n, e, rf, u);
        else load_conv<S, R, NV>(U, n, e, u);
        volume_integral<R, NC, PH, DEV>(P, u, h, rf, res,
                                        (PH == 1 && A.tpt) ? reinterpret_cast<const R *>(A.tpt) + (int64_t) kMemoVolRow * n + e
                                                           : nullptr, n);
        if constexpr (PH == 1) {
            if (A.visc) {
                const S *__restrict__ VI = reinterpret_cast<const S *>(A.visc);
                #pragma unroll
                for (int i = 0; i < 16; i++) res[i] += (R) (VI + i * A.n_elem)[e];
            }
        }
        auto gather = [&](int sl) {
            const int fl = sl >> 1, side = sl & 1;
            const R *m = mom + (size_t) fl * 3 * NV;
            #pragma unroll
            for (int v = 0; v < NV; v++) slot_add<R>(finfo[fl], side, m[v], m[NV + v], m[2 * NV + v], &res[4*v]);
        };
        #pragma unroll
        for (int k = 0; k < 6; k++) gather(sl6[k]);
        for (int si = s_beg + 6; si < s_end; si++) gather(A.slots[si]);
        S *out = reinterpret_cast<S *>(A.out);
        if (A.mode == 0) {
            #pragma unroll
            for (int i = 0; i < 4 * NV; i++) stp<S>(out, n, i, e, (S) res[i]);
        } else {
            // c -= dt * A^-1 int (src/models/euler/charm_model.c:402-433); A^-1
            // of a level-l cube is the FP64 level-0 inverse times 8^l (exact
            // power-of-two scaling), diagonal on the cube octree; then the
            // SSP-RK combine when no limiter sits in between
            // (mixed mode: the stored FP64 coefficient is re-read, the FP32
            // integral widened, and the update and combine run in FP64)
            const S sc = ldexp(S(1), 3 * lev);
            const S dt = S(A.dt);
            // not __restrict__: the last RK stage writes its output over u^n
            const S *U0 = reinterpret_cast<const S *>(A.U0);
            #pragma unroll
            for (int v = 0; v < NV; v++)
                #pragma unroll
                for (int k = 0; k < 4; k++) {
                    const S ai = cst<S>(P.ainv0[k], P.ainv0_f[k]) * sc;
                    // the stored coefficient (the registers hold deviations in DEV)
                    const S uk = (std::is_same<S, R>::value && !DEV) ? (S) u[4*v+k] : ldp<S>(U, n, 4*v+k, e);
                    const S w = uk - dt * (ai * (S) res[4*v+k]);
                    stp<S>(out, n, 4*v+k, e, A.combine ? rk_combine<S>(A.combine, w, ldp<S>(U0, n, 4*v+k, e)) : w);
                }
        }
    }
    if (!ok) A.err[0] = 1;
}

// threads of k_stage_pt's workgroup: five waves take the face and volume
// points of an eight-leaf chunk in one round
constexpr int kPtBlock = 320;

// the flux of face record rec at point k, momentum in global order
template <typename S, typename R, int NC, int FLUX, int PH, bool DEV>
__device__ __forceinline__ bool record_point(const StageArgs &A, const DevParams &P, const S *__restrict__ U, int4 rec,
                                             int k, const DevRef &rf, R *q)
{
    constexpr int NV = 4 + NC;
    const int64_t n = A.n_elem;
    const int dir0 = rec.z & 7, kind = (rec.z >> 3) & 3, sub = (rec.z >> 5) & 3, ax = dir0 >> 1;
    const R g1 = gp_t1<R>(k), g2 = gp_t2<R>(k);
    const R *tl, *tr;
    face_closures<R, PH>(A, rec, tl, tr);
    if (tl) tl += k * n;
    if (tr) tr += k * n;
    const FaceMap<R> fm(kind, sub);
    R ua[4 * NV], o[NV];
    load_frame<S, R, NC, DEV>(U, n, rec.x, ax, rf, ua);
    bool ok;
    if (kind == FACE_BND) {
        const R s = (dir0 & 1) ? R(1) : R(-1);
        DevRef rx = rf;
        mirror_side<R, NV, DEV>(ax, s, ua, rx);
        to_face<R, NV>(R(0.5), ua);
        ok = point_flux<R, NC, FLUX, true, PH, DEV>(P, ua, ua, fm, g1, g2, dir0, s, rx, tl, tr, n, o);
        o[0] *= s;
    } else {
        R ub[4 * NV];
        load_frame<S, R, NC, DEV>(U, n, rec.y, ax, rf, ub);
        to_face<R, NV>(R(0.5), ua);
        to_face<R, NV>(R(-0.5), ub);
        ok = point_flux<R, NC, FLUX, false, PH, DEV>(P, ua, ub, fm, g1, g2, dir0, R(1), rf, tl, tr, n, o);
    }
    const int a = (!DEV || kind == FACE_BND) ? ax : 0;      // DEV: interior fluxes are in global order
    q[0] = a == 0 ? o[0] : o[1];
    q[1] = a == 1 ? o[0] : (a == 0 ? o[1] : o[2]);
    q[2] = a == 2 ? o[0] : o[2];
    #pragma unroll
    for (int v = 3; v < NV; v++) q[v] = o[v];
    return ok;
}

// The stage of a small mesh, one thread per quadrature point.
//
// A mesh of a few thousand leaves does not fill 256 CUs with k_stage's
// chunks: a stage is then the serial chain of one workgroup (three face
// passes of six points each, eight volume points, the gather).  This kernel
// runs a chunk of 8 or 16 leaves with its points spread over the lanes:
//   phase 1  thread = (face, point): both traces and the flux, to LDS;
//            thread = (element, volume point): the volume fluxes, to LDS;
//   phase 2  thread = (face, variable): the three moments over six points;
//   phase 3  thread = (element, variable): the volume sums over eight
//            points, the gather of the face moments, A^-1 and the update.
// The sums run in k_stage's order.  Bound by the chain of dependent loads and
// one point's arithmetic: 22 -> 8 us at 512 leaves (FP64), 21 -> 11 us at
// 4,096 (FP32).  It evaluates 4.9 faces per leaf where k_stage's chunks take
// 3.7, and k_stage wins from about 12,000 leaves on (32,768 leaves, FP32: 36
// against 21 us).
template <typename S, typename R, int NC, int FLUX, int PH>
__global__ __launch_bounds__(kPtBlock)
void k_stage_pt(StageArgs A, DevParams Pv)
{
    const DevParams &P = stage_params<PH>(A, Pv);
    constexpr int NV = 4 + NC, NW = 3 * NV + 1;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const S *__restrict__ U = reinterpret_cast<const S *>(A.U);
    const int c = xcd_block(A.n_xcd);
    if (c >= A.n_chunks) return;                 // whole workgroup exits together
    const int fb = A.ch_fbeg[c], nf = A.ch_fbeg[c + 1] - fb;
    const int eb = A.ch_ebeg[c], ne = A.ch_ebeg[c + 1] - eb;
    const int64_t n = A.n_elem;
    R *fq = reinterpret_cast<R *>(smem_raw);                        // [6][NV][nf] fluxes
    R *mom = fq + 6 * NV * nf;                                      // [nf][3][NV]
    R *vq = mom + 3 * NV * nf;                                      // [8][NW][ne] volume fluxes, density
    int *finfo = reinterpret_cast<int *>(vq + 8 * NW * ne);
    int *flev = finfo + nf;                                         // level of the (small) face
    constexpr bool DEV = uses_dev<R, NC, FLUX, PH>();
    DevRef rf{};
    if constexpr (DEV) rf = chunk_ref<S>(A, P, c);
    bool ok = true;
    // phase 1: face points (point-major, so a wave mostly shares its point),
    // then the volume points from the next whole wave on
    const int np = 6 * nf, vb = (np + 63) & ~63, items = vb + 8 * ne;
    for (int i = (int) threadIdx.x; i < items; i += kPtBlock) {
        if (i < np) {
            const int k = i / nf, f = i - k * nf;
            const int4 rec = A.cf4[fb + f];
            const int kind = (rec.z >> 3) & 3;
            const int lev = A.level[rec.x] + (kind == FACE_HANG1 ? 1 : 0);
            R q[NV];
            ok &= record_point<S, R, NC, FLUX, PH, DEV>(A, P, U, rec, k, rf, q);
            #pragma unroll
            for (int v = 0; v < NV; v++) fq[(k * NV + v) * nf + f] = q[v];
            if (k == 0) { finfo[f] = rec.z; flev[f] = lev; }
        } else if (i >= vb) {
            const int g = (i - vb) / ne, el = (i - vb) - g * ne;
            R u[4 * NV], F[3][NV];
            if constexpr (DEV) load_dev<S>(U, n, eb + el, rf, u);
            else load_conv<S, R, NV>(U, n, eb + el, u);
            const R *tk = (PH == 1 && A.tpt) ? reinterpret_cast<const R *>(A.tpt) + (int64_t) (kMemoVolRow + g) * n + eb + el
                                             : nullptr;
            const R r = volume_terms<R, NC, PH, DEV>(P, u, g, rf, tk, n, F);
            #pragma unroll
            for (int d = 0; d < 3; d++)
                #pragma unroll
                for (int v = 0; v < NV; v++) vq[(g * NW + d * NV + v) * ne + el] = F[d][v];
            vq[(g * NW + 3 * NV) * ne + el] = r;
        }
    }
    __syncthreads();
    for (int i = (int) threadIdx.x; i < NV * nf; i += kPtBlock) {
        const int v = i / nf, f = i - v * nf;
        const R h = ldexp(R(1), -flev[f]), wj = h * h * R(1.0 / 6.0);
        R s0 = R(0), s1 = R(0), s2 = R(0);
        #pragma unroll
        for (int k = 0; k < 6; k++) {
            const R q = fq[(k * NV + v) * nf + f];
            s0 += q; s1 = fma(q, gp_t1<R>(k), s1); s2 = fma(q, gp_t2<R>(k), s2);
        }
        R *m = mom + (size_t) f * 3 * NV + v;
        m[0] = s0 * wj; m[NV] = s1 * wj; m[2 * NV] = s2 * wj;
    }
    __syncthreads();
    for (int i = (int) threadIdx.x; i < NV * ne; i += kPtBlock) {
        const int v = i / ne, el = i - v * ne, e = eb + el;
        const int lev = A.level[e];
        const R h = ldexp(R(1), -lev), hinv = rcp(h), wv = h * h * h * R(0.125), fv = wv * hinv;
        R res[4];
        {
            R sf[3] = {R(0), R(0), R(0)};
            #pragma unroll
            for (int g = 0; g < 8; g++)
                #pragma unroll
                for (int d = 0; d < 3; d++) sf[d] += vq[(g * NW + d * NV + v) * ne + el];
            res[0] = R(0); res[1] = -sf[0] * fv; res[2] = -sf[1] * fv; res[3] = -sf[2] * fv;
        }
        if (v < 3) {
            const R ph = R(0.28867513459481288225);
            const R gv = v == 0 ? cst<R>(P.grav[0], P.grav_f[0]) : (v == 1 ? cst<R>(P.grav[1], P.grav_f[1])
                                                                            : cst<R>(P.grav[2], P.grav_f[2]));
            R G[4] = {R(0), R(0), R(0), R(0)};
            #pragma unroll
            for (int g = 0; g < 8; g++) {
                const R r = vq[(g * NW + 3 * NV) * ne + el];
                G[0] += r; G[1] += r * ((g & 1) ? ph : -ph); G[2] += r * ((g & 2) ? ph : -ph);
                G[3] += r * ((g & 4) ? ph : -ph);
            }
            #pragma unroll
            for (int k = 0; k < 4; k++) res[k] -= gv * G[k] * wv;
        }
        if constexpr (PH == 1) {
            if (A.visc && v < 4) {
                const S *__restrict__ VI = reinterpret_cast<const S *>(A.visc);
                #pragma unroll
                for (int k = 0; k < 4; k++) res[k] += (R) (VI + (int64_t) (4 * v + k) * n)[e];
            }
        }
        const int s_end = A.slot_ptr[e + 1];
        for (int si = A.slot_ptr[e]; si < s_end; si++) {
            const int sl = A.slots[si], fl = sl >> 1, side = sl & 1;
            const R *m = mom + (size_t) fl * 3 * NV + v;
            slot_add<R>(finfo[fl], side, m[0], m[NV], m[2 * NV], res);
        }
        // the update of k_stage for one variable
        S *out = reinterpret_cast<S *>(A.out);
        const S *U0 = reinterpret_cast<const S *>(A.U0);
        const S sc = ldexp(S(1), 3 * lev), dt = S(A.dt);
        #pragma unroll
        for (int k = 0; k < 4; k++) {
            const int64_t at = (int64_t) (4 * v + k) * n + e;
            if (A.mode == 0) { out[at] = (S) res[k]; continue; }
            const S ai = cst<S>(P.ainv0[k], P.ainv0_f[k]) * sc;
            const S w = U[at] - dt * (ai * (S) res[k]);
            out[at] = A.combine ? rk_combine<S>(A.combine, w, U0[at]) : w;
        }
    }
    if (!ok) A.err[0] = 1;
}

template <typename S, typename R, int NC, int PH>
static hipError_t launch_stage_pt(int flux, const StageArgs &A, const DevParams &P, hipStream_t st)
{
    const size_t sh = stage_points_smem_bytes(sizeof(R) == 4, NC, A.max_faces, A.chunk_elems);
    const dim3 grid((unsigned) (((A.n_chunks + A.n_xcd - 1) / A.n_xcd) * A.n_xcd)), block(kPtBlock);
    switch (flux) {
    case FLUX_LF: hipLaunchKernelGGL((k_stage_pt<S, R, NC, FLUX_LF, PH>), grid, block, sh, st, A, P); break;
    case FLUX_HLLC: hipLaunchKernelGGL((k_stage_pt<S, R, NC, FLUX_HLLC, PH>), grid, block, sh, st, A, P); break;
    case FLUX_GODUNOV: hipLaunchKernelGGL((k_stage_pt<S, R, NC, FLUX_GODUNOV, PH>), grid, block, sh, st, A, P); break;
    case FLUX_CD: hipLaunchKernelGGL((k_stage_pt<S, R, NC, FLUX_CD, PH>), grid, block, sh, st, A, P); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename S, typename R, int NC, int BS, int PH>
static hipError_t launch_stage_bs(int flux, const StageArgs &A, const DevParams &P, hipStream_t st)
{
    constexpr int NV = 4 + NC;
    if (A.points) return launch_stage_pt<S, R, NC, PH>(flux, A, P, st);
    const size_t sh = (size_t) A.max_faces * (3 * NV * sizeof(R) + sizeof(int));
    const dim3 grid((unsigned) (((A.n_chunks + A.n_xcd - 1) / A.n_xcd) * A.n_xcd)), block(BS);
    switch (flux) {
    case FLUX_LF: hipLaunchKernelGGL((k_stage<S, R, NC, FLUX_LF, BS, PH>), grid, block, sh, st, A, P); break;
    case FLUX_HLLC: hipLaunchKernelGGL((k_stage<S, R, NC, FLUX_HLLC, BS, PH>), grid, block, sh, st, A, P); break;
    case FLUX_GODUNOV:
        if constexpr (sizeof(R) == 8 && NC == 2 && PH == 0) {
            if (A.n_elem > 100000) {
                hipLaunchKernelGGL((k_stage<S, R, NC, FLUX_GODUNOV, BS, PH, 2>), grid, block, sh, st, A, P);
                break;
            }
        }
        hipLaunchKernelGGL((k_stage<S, R, NC, FLUX_GODUNOV, BS, PH>), grid, block, sh, st, A, P);
        break;
    case FLUX_CD: hipLaunchKernelGGL((k_stage<S, R, NC, FLUX_CD, BS, PH>), grid, block, sh, st, A, P); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// host address of one stage kernel instance (for its attributes)
template <typename S, typename R, int NC, int BS, int PH>
static const void *stage_fn_bs(int flux)
{
    switch (flux) {
    case FLUX_LF: return reinterpret_cast<const void *>(&k_stage<S, R, NC, FLUX_LF, BS, PH>);
    case FLUX_HLLC: return reinterpret_cast<const void *>(&k_stage<S, R, NC, FLUX_HLLC, BS, PH>);
    case FLUX_GODUNOV: return reinterpret_cast<const void *>(&k_stage<S, R, NC, FLUX_GODUNOV, BS, PH>);
    case FLUX_CD: return reinterpret_cast<const void *>(&k_stage<S, R, NC, FLUX_CD, BS, PH>);
    }
    return nullptr;
}

template <typename S, typename R, int PH>
const void *stage_fn_t(int nc, int flux, int bs)
{
    const bool wide = PH == 1 || bs > 128;
    switch (nc) {
    case 1: return wide ? stage_fn_bs<S, R, 1, 256, PH>(flux) : stage_fn_bs<S, R, 1, 128, PH>(flux);
    case 2: return wide ? stage_fn_bs<S, R, 2, 256, PH>(flux) : stage_fn_bs<S, R, 2, 128, PH>(flux);
    case 3: return wide ? stage_fn_bs<S, R, 3, 256, PH>(flux) : stage_fn_bs<S, R, 3, 128, PH>(flux);
    case 4: return wide ? stage_fn_bs<S, R, 4, 256, PH>(flux) : stage_fn_bs<S, R, 4, 128, PH>(flux);
    }
    return nullptr;
}

// one thread per chunk element: 128- or 256-element chunks (the
// Navier-Stokes variant always runs 256-thread workgroups)
template <typename S, typename R, int PH>
hipError_t launch_stage_t(int nc, int flux, const StageArgs &A, const DevParams &P, hipStream_t st)
{
    if (A.chunk_elems > 256) return hipErrorInvalidValue;
    if constexpr (PH == 1) {
        switch (nc) {
        case 1: return launch_stage_bs<S, R, 1, 256, PH>(flux, A, P, st);
        case 2: return launch_stage_bs<S, R, 2, 256, PH>(flux, A, P, st);
        case 3: return launch_stage_bs<S, R, 3, 256, PH>(flux, A, P, st);
        case 4: return launch_stage_bs<S, R, 4, 256, PH>(flux, A, P, st);
        }
        return hipErrorInvalidValue;
    } else {
        const bool wide = A.block > 128;
        switch (nc) {
        case 1: return wide ? launch_stage_bs<S, R, 1, 256, PH>(flux, A, P, st) : launch_stage_bs<S, R, 1, 128, PH>(flux, A, P, st);
        case 2: return wide ? launch_stage_bs<S, R, 2, 256, PH>(flux, A, P, st) : launch_stage_bs<S, R, 2, 128, PH>(flux, A, P, st);
        case 3: return wide ? launch_stage_bs<S, R, 3, 256, PH>(flux, A, P, st) : launch_stage_bs<S, R, 3, 128, PH>(flux, A, P, st);
        case 4: return wide ? launch_stage_bs<S, R, 4, 256, PH>(flux, A, P, st) : launch_stage_bs<S, R, 4, 128, PH>(flux, A, P, st);
        }
        return hipErrorInvalidValue;
    }
}

} // namespace charm
