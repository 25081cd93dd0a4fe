// march.hpp -- the fused MUSCL-Hancock + Riemann + Godunov step kernel (k_step_march) and
// the per-cell helpers it shares with the ghost-fill and CFL kernels.
//
// Design (gfx950):
//  * The grid is cut into in-plane tiles (x in 2D; x-y in 3D) and segments
//    along the last active dim (the "march" dim).  A workgroup owns one tile
//    plus a one-cell halo ring ("Hancock region", one thread per column) and
//    marches through its segment one plane at a time.
//  * Per plane h: each column loads the conservative state at h+1, converts
//    to primitives, publishes plane h's primitives (plus a two-cell ring) in
//    LDS, reconstructs all faces (limited slopes along every dim: in-plane
//    neighbours from LDS, march neighbours from registers), converts the face
//    states to conservative form and applies the Hancock half step -- the
//    reference's face_reconstruction / conv_prim_to_cons / Hancock kernels for
//    one cell, in registers.
//  * In-plane faces: the right neighbour solves the Riemann problem once per
//    face; x face states and fluxes pass between lanes, y ones through LDS.  March-dim faces: the right face state of
//    plane h-1 is kept in registers and paired with plane h's left state.
//  * The Godunov update of a cell accumulates dims in the reference order
//    (flux, geometric sources, gravity per dim, march dim last), so with the
//    FP64 policy every conserved value is bit-identical to the reference's
//    unfused sequence (down to the range of physics.hpp fdiv: values below
//    about 1e-290 may differ in their last bits).
//  * Face states never touch HBM: per cell-update the kernel reads the
//    conservative state once (plus halo re-reads served mostly by L2) and
//    writes it once.  The epilogue reduces (in FP64) the CFL rate of the new
//    state, the minimum internal energy of the consumed state and the
//    conserved totals; per-workgroup partials are folded in a fixed order.
//  * The kernels are generic over the precision policy (physics.hpp):
//    PerfectGas streams FP64; PerfectGasMixed streams FP32 (half the bytes)
//    with FP64 pressure recovery and FP64 reductions; PerfectGasFast streams
//    FP64 with the reference's formulas evaluated without its rounding.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fused.hpp"
#include "launch.hpp"
#include "physics.hpp"
#include "pressure_fix.hpp"
#include "reduce.hpp"

namespace hclpp {

template <int ND>
__device__ __forceinline__ int64_t cell_at(const GridDev& G, int a, int b, int m)
{
    if constexpr (ND == 1) return (int64_t)m;
    else if constexpr (ND == 2) return (int64_t)a + (int64_t)G.nwg[0] * (int64_t)m;
    else return flat(G, a, b, m);
}

template <int ND>
__device__ __forceinline__ void ijk_of(int a, int b, int m, int& i, int& j, int& k)
{
    if constexpr (ND == 1) { i = m; j = 0; k = 0; }
    else if constexpr (ND == 2) { i = a; j = m; k = 0; }
    else { i = a; j = b; k = m; }
}

// Register exchange with the neighbouring column along x.  A tile row of ROW columns occupies
// ROW consecutive lanes (3D: 16, a DPP row, row_shr / row_shl; 2D: 64, the whole wave, wave_shr /
// wave_shl), so the column at x - 1 (FROM_LEFT) or x + 1 is the lane beside this one.  Every lane
// of the wave must execute the shift; the first (FROM_LEFT) or last lane of a row receives 0.
template <int ROW, bool FROM_LEFT>
__device__ __forceinline__ int lane_shift_u32(int v)
{
    static_assert(ROW == 16 || ROW == 64, "tile rows of 16 or 64 columns");
    constexpr int kCtrl = ROW == 16 ? (FROM_LEFT ? 0x111 : 0x101) : (FROM_LEFT ? 0x138 : 0x130);
    return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xF, 0xF, true);
}

template <int ROW, bool FROM_LEFT>
__device__ __forceinline__ double lane_shift(double v)
{
    int2 p = __builtin_bit_cast(int2, v);
    p.x = lane_shift_u32<ROW, FROM_LEFT>(p.x);
    p.y = lane_shift_u32<ROW, FROM_LEFT>(p.y);
    return __builtin_bit_cast(double, p);
}

template <int ROW, bool FROM_LEFT>
__device__ __forceinline__ float lane_shift(float v)
{
    return __builtin_bit_cast(float, lane_shift_u32<ROW, FROM_LEFT>(__builtin_bit_cast(int, v)));
}

template <int ND, class S>
__device__ __forceinline__ State<ND, S> load_cons(const StepArraysT<S>& A, const GridDev& G, int64_t id)
{
    State<ND, S> c;
    c[0] = A.rho[id];
#pragma unroll
    for (int d = 0; d < ND; ++d) c[1 + d] = A.rhou[id + G.plane * d];
    c[ND + 1] = A.E[id];
    return c;
}

template <int ND, class S>
__device__ __forceinline__ void store_cons(const StepArraysT<S>& A, const GridDev& G, int64_t id, const State<ND, S>& c)
{
    A.rho_new[id] = c[0];
#pragma unroll
    for (int d = 0; d < ND; ++d) A.rhou_new[id + G.plane * d] = c[1 + d];
    A.E_new[id] = c[ND + 1];
}

// CFL rate of a conservative state at (i,j,k) (time_step.hpp:61-76), in FP64.  With the
// FP64 policies this is the policy's conv_cons_to_prim, then the rate (the reference's
// arithmetic for PerfectGas).
template <int ND, int GEOM, class Eos>
__device__ __forceinline__ double state_rate(const GridDev& G, const Eos& eos, int i, int j, int k, const State<ND, typename Eos::real>& c)
{
    if constexpr (kFp64State<Eos>) {
        double evol, y, cs;
        State<ND> const p = cons_to_prim_ey(c, eos, evol, y);
        if constexpr (std::is_same_v<Eos, PerfectGas>) cs = eos.sound(p[0], p[ND + 1], y);
        else cs = eos.sound(p[0], p[ND + 1]);
        return cfl_rate<ND, GEOM>(G, i, j, k, &p.q[1], cs);
    } else {
        double const rho = c[0];
        double u[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) u[d] = fdiv((double)c[1 + d], rho);
        double const P = eos.gamma_m1 * eos.internal_energy_fp64(c);
        return cfl_rate<ND, GEOM>(G, i, j, k, u, sqrt(fdiv(eos.gamma_d * P, rho)));
    }
}

// Internal energy E - |m|^2 / 2 rho of a conservative state in FP64 (internal_energy.cpp:25-40).
template <int ND, class Eos>
__device__ __forceinline__ double state_eint(const Eos& eos, const State<ND, typename Eos::real>& c)
{
    if constexpr (std::is_same_v<Eos, PerfectGas>) return internal_energy(c);
    else return eos.internal_energy_fp64(c);
}

// The distances of a cell's center to its neighbours' along one dim, with their reciprocals
// (GridDev::hc): (dx[i-1] + dx[i]) / 2 and (dx[i] + dx[i+1]) / 2.  With FP32 state the distances are FP32
// sums and the reciprocals v_rcp_f32's, as PerfectGasMixed::div takes them: rounding the table's
// instead moves a blast wave's far field by 1e-5.
struct CenterDist {
    double hm, ym, hp, yp;
};
template <class Eos>
__device__ __forceinline__ CenterDist center_dist(const GridDev& G, int dim, int i)
{
    if constexpr (kFp64State<Eos>) {
        double const* h = G.hc[dim] + 2 * (i - 1);
        return {h[0], h[1], h[2], h[3]};
    } else {
        float const dl = (float)G.dx[dim][i];
        float const hm = ((float)G.dx[dim][i - 1] + dl) * 0.5f, hp = (dl + (float)G.dx[dim][i + 1]) * 0.5f;
        return {hm, __builtin_amdgcn_rcpf(hm), hp, __builtin_amdgcn_rcpf(hp)};
    }
}

// limited_linear_reconstruction.hpp:53-62 for one variable along one dim
template <int LIM, class Eos, class T>
__device__ __forceinline__ void reconstruct(T vm, T v, T vp, const CenterDist& h, T dl, T& lo, T& hi)
{
    T const slope = slope_limiter<LIM, Eos, T>(Eos::quot_grid(vp - v, h.hp, h.yp), Eos::quot_grid(v - vm, h.hm, h.ym));
    lo = v - ((dl * T(0.5)) * slope);
    hi = v + ((dl * T(0.5)) * slope);
}

// Spherical sources of one dim for the cell's own face states (godunov_scheme.hpp:165-256),
// applied to the accumulator in the reference order.  pL and pR are the primitives of those
// states, which the Riemann solves of the two faces have formed.
template <class Eos, int ND, int GEOM>
__device__ __forceinline__ void godunov_sources(const GridDev& G, int dim, int i, int j, typename Eos::real dtodv,
                                                typename Eos::real dS, typename Eos::real dSp, const State<ND, typename Eos::real>& pL,
                                                const State<ND, typename Eos::real>& pR, State<ND, typename Eos::real>& un)
{
    using T = typename Eos::real;
    if constexpr (GEOM == kSpherical) {
        if (dim > 1) return;
        T const x0 = T(G.x[0][i]), x0p = T(G.x[0][i + 1]);
        if (dim == 0) {
            un[1] += src_pressure<Eos>(dtodv, pL[ND + 1], pR[ND + 1], dS, dSp);
            if constexpr (ND >= 2) {
                un[1] += src_centrifugal<Eos>(dtodv, pL[0], pR[0], pL[2], pR[2], dS, dSp);
                un[2] -= src_coriolis_r<Eos>(dtodv, x0, x0p, pL[0], pR[0], pL[1], pR[1], pL[2], pR[2], dS, dSp);
            }
            if constexpr (ND == 3) {
                un[1] += src_centrifugal<Eos>(dtodv, pL[0], pR[0], pL[3], pR[3], dS, dSp);
                un[3] -= src_coriolis_r<Eos>(dtodv, x0, x0p, pL[0], pR[0], pL[1], pR[1], pL[3], pR[3], dS, dSp);
            }
        } else {
            un[2] += src_pressure<Eos>(dtodv, pL[ND + 1], pR[ND + 1], dS, dSp);
            if constexpr (ND == 3) {
                un[2] += src_centrifugal_th<Eos>(dtodv, T(G.cot_mid[j]), pL[0], pR[0], pL[3], pR[3], dS, dSp);
                un[3] -= src_coriolis_th<Eos>(dtodv, T(G.sin_node[j]), T(G.sin_node[j + 1]), pL[0], pR[0], pL[2], pR[2], pL[3], pR[3], dS,
                                              dSp);
            }
        }
    }
}

// Passive scalars of one cell or face (mass fractions, or partial densities during an update);
// a one-slot placeholder when the step has none.
template <int NFX, class T>
struct Frac {
    T f[NFX > 0 ? NFX : 1];
};

template <int NFX, class T>
__device__ __forceinline__ Frac<NFX, T> zero_frac()
{
    Frac<NFX, T> x;
#pragma unroll
    for (int f = 0; f < (NFX > 0 ? NFX : 1); ++f) x.f[f] = 0;
    return x;
}

// MUSCL-Hancock predictor of one cell (hydro_reconstruction.hpp:99-128 and
// extrapolation_reconstruction.hpp:90-337): nb[dim][side] are the primitive
// neighbours (side 0 = minus, 1 = plus) along each dim; x and xnb the passive
// scalars of the cell and of the same neighbours, xf their face values after the
// half step (mass fractions, as fx_rec leaves the predictor).
template <class Eos, int ND, int GEOM, int LIM, int NFX>
__device__ __forceinline__ void predict_faces(const GridDev& G, const Eos& eos, typename Eos::real dth, typename Eos::real dtodv, int i, int j, int k,
                                              const State<ND, typename Eos::real>& p, const State<ND, typename Eos::real> (&nb)[ND][2],
                                              State<ND, typename Eos::real> (&fs)[2][ND], const Frac<NFX, typename Eos::real>& x,
                                              const Frac<NFX, typename Eos::real> (&xnb)[ND][2], Frac<NFX, typename Eos::real> (&xf)[2][ND])
{
    using T = typename Eos::real;
    constexpr int NV = ND + 2;
    State<ND, T> fp[2][ND];
    Frac<NFX, T> xo[2][ND];  // reconstructed mass fractions, kept for the scalar fluxes (extrapolation_reconstruction.hpp:87-88)
    int const idx[3] = {i, j, k};
#pragma unroll
    for (int dim = 0; dim < ND; ++dim) {
        T const dl = T(G.dx[dim][idx[dim]]);
        CenterDist const h = center_dist<Eos>(G, dim, idx[dim]);
#pragma unroll
        for (int v = 0; v < NV; ++v)
            reconstruct<LIM, Eos>(nb[dim][0][v], p[v], nb[dim][1][v], h, dl, fp[0][dim][v], fp[1][dim][v]);
        if constexpr (NFX > 0) {
#pragma unroll
            for (int f = 0; f < NFX; ++f)
                reconstruct<LIM, Eos>(xnb[dim][0].f[f], x.f[f], xnb[dim][1].f[f], h, dl, xo[0][dim].f[f], xo[1][dim].f[f]);
        }
    }
#pragma unroll
    for (int dim = 0; dim < ND; ++dim)
#pragma unroll
        for (int s = 0; s < 2; ++s) fs[s][dim] = prim_to_cons(fp[s][dim], eos);
    T rho_old[2][ND], mom_old[2][ND][ND], E_face[2][ND];
#pragma unroll
    for (int dim = 0; dim < ND; ++dim)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            rho_old[s][dim] = fs[s][dim][0];
            E_face[s][dim] = fs[s][dim][ND + 1];  // the face's total energy, reused by its flux
#pragma unroll
            for (int v = 0; v < ND; ++v) mom_old[s][dim][v] = fs[s][dim][1 + v];
        }
    if constexpr (NFX > 0) {  // extrapolation_reconstruction.hpp:105-108: partial densities of the faces
#pragma unroll
        for (int dim = 0; dim < ND; ++dim)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int f = 0; f < NFX; ++f) xf[s][dim].f[f] = xo[s][dim].f[f] * rho_old[s][dim];
    }
    T const x0 = T(G.x[0][i]), x0p = T(G.x[0][i + 1]);
#pragma unroll
    for (int dim = 0; dim < ND; ++dim) {
        State<ND, T> const& pL = fp[0][dim];
        State<ND, T> const& pR = fp[1][dim];
        State<ND, T> const fL = flux_of_prim_e<ND, T>(pL, dim, E_face[0][dim]);
        State<ND, T> const fR = flux_of_prim_e<ND, T>(pR, dim, E_face[1][dim]);
        T const dS = T(face_area<ND, GEOM>(G, dim, i, j, k));
        T const dSp = T(face_area<ND, GEOM>(G, dim, i + (dim == 0), j + (dim == 1), k + (dim == 2)));
#pragma unroll
        for (int pos = 0; pos < ND; ++pos)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int v = 0; v < NV; ++v) fs[s][pos][v] += dtodv * ((fL[v] * dS) - (fR[v] * dSp));
        if constexpr (GEOM == kSpherical) {
#pragma unroll
            for (int pos = 0; pos < ND; ++pos)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (dim == 0) {
                        fs[s][pos][1] += src_pressure<Eos>(dtodv, pL[ND + 1], pR[ND + 1], dS, dSp);
                        if constexpr (ND >= 2) {
                            fs[s][pos][1] += src_centrifugal<Eos>(dtodv, pL[0], pR[0], pL[2], pR[2], dS, dSp);
                            fs[s][pos][2] -= src_coriolis_r<Eos>(dtodv, x0, x0p, pL[0], pR[0], pL[1], pR[1], pL[2], pR[2], dS, dSp);
                        }
                        if constexpr (ND == 3) {
                            fs[s][pos][1] += src_centrifugal<Eos>(dtodv, pL[0], pR[0], pL[3], pR[3], dS, dSp);
                            fs[s][pos][3] -= src_coriolis_r<Eos>(dtodv, x0, x0p, pL[0], pR[0], pL[1], pR[1], pL[3], pR[3], dS, dSp);
                        }
                    }
                    if (dim == 1) {
                        fs[s][pos][2] += src_pressure<Eos>(dtodv, pL[ND + 1], pR[ND + 1], dS, dSp);
                        if constexpr (ND == 3) {
                            fs[s][pos][2] += src_centrifugal_th<Eos>(dtodv, T(G.cot_mid[j]), pL[0], pR[0], pL[3], pR[3], dS, dSp);
                            fs[s][pos][3] -= src_coriolis_th<Eos>(dtodv, T(G.sin_node[j]), T(G.sin_node[j + 1]), pL[0], pR[0], pL[2], pR[2],
                                                                  pL[3], pR[3], dS, dSp);
                        }
                    }
                }
        }
        if (gravity_acts(G, dim)) {
            T const g = T(gravity(G, i, dim));
#pragma unroll
            for (int pos = 0; pos < ND; ++pos)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    fs[s][pos][1 + dim] += dth * g * rho_old[s][pos];
                    fs[s][pos][ND + 1] += dth * g * mom_old[s][pos][dim];
                }
        }
        if constexpr (NFX > 0) {  // extrapolation_reconstruction.hpp:315-323
#pragma unroll
            for (int f = 0; f < NFX; ++f) {
                T const ffL = xo[0][dim].f[f] * fL[0];
                T const ffR = xo[1][dim].f[f] * fR[0];
#pragma unroll
                for (int pos = 0; pos < ND; ++pos)
#pragma unroll
                    for (int s = 0; s < 2; ++s) xf[s][pos].f[f] += dtodv * ((ffL * dS) - (ffR * dSp));
            }
        }
    }
    if constexpr (NFX > 0) {  // passive_scalar_extrapolation (extrapolation_reconstruction.hpp:327-337)
#pragma unroll
        for (int dim = 0; dim < ND; ++dim)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int f = 0; f < NFX; ++f) xf[s][dim].f[f] = Eos::div(xf[s][dim].f[f], fs[s][dim][0]);
    }
}

// The columns of a march workgroup.  Workgroup b of nb owns a tile of columns (3D: HX x HY, 2D: a
// row of HX, 1D: NT segments of one column) and a segment of planes of the march dim; thread tid
// owns column (a, bb) (ghost-inclusive coordinates of the in-plane dims; a tile's first and last
// columns are halo) and planes [zs, ze).  Blocks that share an XCD (b % 8) get consecutive tiles,
// so halo re-reads hit that XCD's L2.
struct MarchColumn {
    int hx, hy, ox, oy, a, bb, zs, ze;
    bool out_col;  // the column holds output cells
    bool seg_ok;   // the segment holds planes (1D: a thread may have none)
};

template <int ND, int HX, int HY, int NT>
__device__ __forceinline__ MarchColumn march_column(const GridDev& G, const FusedLayout& L, int b, int nb, int tid)
{
    constexpr int MD = ND - 1;
    constexpr int TX = (ND >= 2) ? HX - 2 : 1;
    constexpr int TY = (ND == 3) ? HY - 2 : 1;
    MarchColumn c{};
    int const q = nb / 8, rem = nb % 8, x8 = b % 8;
    int const lb = x8 * q + (x8 < rem ? x8 : rem) + b / 8;
    int seg;
    if constexpr (ND == 1) {
        seg = lb * NT + tid;
    } else {
        c.hx = tid % HX;
        c.hy = tid / HX;
        int const tx = lb % L.ntile[0];
        int const rest = lb / L.ntile[0];
        int const ty = rest % L.ntile[1];
        seg = rest / L.ntile[1];
        c.ox = G.ngh[0] + tx * TX;
        c.oy = (ND == 3) ? G.ngh[1] + ty * TY : 0;
    }
    c.a = c.ox - 1 + c.hx;
    c.bb = (ND == 3) ? c.oy - 1 + c.hy : 0;
    int const ngm = G.ngh[MD], nm = G.n[MD];
    c.zs = ngm + seg * L.seglen;
    c.ze = min(c.zs + L.seglen, ngm + nm);
    c.seg_ok = c.zs < ngm + nm;
    c.out_col = c.seg_ok;
    if constexpr (ND >= 2) c.out_col = c.out_col && c.hx >= 1 && c.hx <= TX && c.a < G.ngh[0] + G.n[0];
    if constexpr (ND == 3) c.out_col = c.out_col && c.hy >= 1 && c.hy <= TY && c.bb < G.ngh[1] + G.n[1];
    return c;
}

// Minimum waves per SIMD the register allocator must allow.  Measured on MI355X: the 3D
// FP32-storage kernel gains 23 % at 3 waves (168 VGPRs); the 3D FP64 kernels gain 30 % at 2 waves
// (256 VGPRs, with the LDS parking below; two workgroups fit a CU's LDS): RT 256^3 runs without a
// spill, spherical Sedov with 12 spilled registers at 7.6 Gcell/s against 5.7 at one wave.  With a
// passive scalar the spherical FP64 kernel spills 79 registers there and loses a third.  The 2D
// kernels lose when forced above their natural 2 or 4.
template <class Eos, int ND, int GEOM, int NFX>
constexpr int march_min_waves()
{
    if constexpr (ND != 3) return 1;
    else if constexpr (!kFp64State<Eos>) return 3;
    else return GEOM == kSpherical && NFX > 0 ? 1 : 2;
}

// NFX of a k_step_march that carries no scalars but stores the mass flux through every face
// (StepArraysT::mflux), for the scalar kernel that follows it (scalar_march.hpp).
constexpr int kStoreMass = -1;

// Load the NFX passive scalars (mass fractions, layout [f][cell]) of one cell.
template <int NFX, class S>
__device__ __forceinline__ Frac<NFX, S> load_frac(const StepArraysT<S>& A, const GridDev& G, int64_t id)
{
    Frac<NFX, S> x;
#pragma unroll
    for (int f = 0; f < NFX; ++f) x.f[f] = A.fx[id + G.plane * f];
    return x;
}

// NFX: passive scalars carried through the step (0, or 1 for the kernels of step_fused_fx.hip), or
// kStoreMass.
template <class Eos, int ND, int GEOM, int RS, int LIM, int NFX, int HX, int HY, int NT>
__global__ __launch_bounds__(NT, (march_min_waves<Eos, ND, GEOM, NFX>())) void k_step_march(GridDev G, Eos eos, StepArraysT<typename Eos::real> A, FusedLayout L)
{
    using T = typename Eos::real;
    using X = Frac<NFX, T>;
    constexpr int NV = ND + 2;
    constexpr int NS = NFX > 0 ? NFX : 0;    // scalars carried
    constexpr int NL = NV + NS;              // values per column in the LDS planes
    constexpr int NP = ND - 1;               // in-plane dims
    constexpr int MD = ND - 1;               // march dim
    constexpr int PX = (ND >= 2) ? HX + 2 : 1;
    constexpr int PY = (ND == 3) ? HY + 2 : 1;
    constexpr int TX = (ND >= 2) ? HX - 2 : 1;
    constexpr int TY = (ND == 3) ? HY - 2 : 1;
    constexpr int NXCH = NP > 0 ? NP : 1;
    // Barriers per plane: one after the primitive plane (double-buffered by plane parity) and, in
    // 3D, one after the y face states and one after the y fluxes.  The y face states take the
    // primitive buffer of the other parity (its plane is read out by then) and the fluxes a buffer
    // of their own, so no write waits for the readers of the previous plane's buffer beyond the
    // barrier that already separates them.  x faces are exchanged between lanes (lane_shift), not
    // through LDS.
    __shared__ T s_prim[2][NL][PY][PX];
    __shared__ T s_fl[ND == 3 ? NL : 1][ND == 3 ? HY : 1][ND == 3 ? HX : 1];
    // 3D spherical: the primitives a column's right y face gets in its neighbour's Riemann solve
    // (velocities along y and z, pressure), which the column's geometric sources read; forming them
    // again costs a state conversion per face (Sedov 7.15 -> 7.4 Gcell/s without)
    constexpr bool kFaceP = ND == 3 && GEOM == kSpherical;
    __shared__ T s_fp[kFaceP ? NV - 2 : 1][kFaceP ? HY : 1][kFaceP ? HX : 1];
    __shared__ double s_red[NT / 64];
    // Per-thread parking of the values plane h-1 hands to plane h (its right march face state,
    // its partial update and its left march flux, and the scalar's): written at the end of a
    // plane, read back when plane h completes plane h-1.  Only the owning thread touches its
    // slots, so no barrier is involved, and the registers are free across the plane's
    // arithmetic.  3D only: in 2D it gained nothing.
    constexpr bool kPark = ND == 3 && !(NFX > 0 && kFp64State<Eos> && GEOM == kSpherical);
    constexpr int NPARK = kPark ? 3 * NV + 3 * NS : 1;
    __shared__ T s_park[NPARK][kPark ? NT : 1];

    DevClock const* clk = A.clock;
    if (clk->pub.done || clk->pub.status) return;
    double const dt_d = clk->pub.dt;
    double const dth_d = dt_d / 2;
    T const dt = T(dt_d);
    T const dth = T(dth_d);

    int const tid = threadIdx.x;
    MarchColumn const mc = march_column<ND, HX, HY, NT>(G, L, blockIdx.x, gridDim.x, tid);
    int const hx = mc.hx, hy = mc.hy, ox = mc.ox, oy = mc.oy, zs = mc.zs, ze = mc.ze;
    bool const out_col = mc.out_col, seg_ok = mc.seg_ok;
    // Columns of a ragged last tile that lie beyond the array repeat its last column, so every lane
    // runs the same code on a valid state and no value is selected around it: only the columns that
    // hold output cells store, reduce or are read by one that does.  (With a branch around each part
    // that a column may not need the compiler kept a second, initialised copy of every result of it:
    // 70 register moves per plane of the 3D kernel, 3 % of its time.)
    int const a = ND >= 2 ? min(mc.a, G.nwg[0] - 1) : 0, bb = ND == 3 ? min(mc.bb, G.nwg[1] - 1) : 0;
    // kStoreMass: the faces whose fluxes this column stores, below its output cells and, from the
    // column (row) past the last one, above the last output cell
    bool const in_x = hx >= 1 && hx <= TX && mc.a < G.ngh[0] + G.n[0];
    bool const in_y = ND < 3 || (hy >= 1 && hy <= TY && mc.bb < G.ngh[1] + G.n[1]);
    bool const x_face = NFX == kStoreMass && ND >= 2 && in_y && (in_x || (hx >= 1 && mc.a == G.ngh[0] + G.n[0]));
    bool const y_face = NFX == kStoreMass && ND == 3 && in_x && (in_y || (hy >= 1 && mc.bb == G.ngh[1] + G.n[1]));
    // Waves of a 3D tile all of whose rows lie beyond the last row that needs a predictor (bb = ngh + n)
    // only keep the barriers.
    static_assert(ND == 1 || NT == HX * HY, "one thread per column of the tile");
    bool const live = ND < 3 || oy - 1 + __builtin_amdgcn_readfirstlane(hy) <= G.ngh[1] + G.n[1];

    // ring cells of the primitive plane (in-plane distance 2 from the output tile)
    constexpr int NRING = (ND == 3) ? 2 * (PX - 2) + 2 * (PY - 2) : ((ND == 2) ? 2 : 0);

    double r_inv = reduce_identity<kMax>();
    double r_emin = reduce_identity<kMin>();
    double r_sum[NV];
    // 3D spherical FP64 (256 registers): four of the conserved totals live in LDS (the thread's own
    // slots) instead of in registers across the march, as many as two workgroups per CU leave room
    // for (Sedov 7.0 -> 7.4 Gcell/s)
    constexpr int kSumLds = kPark && kFp64State<Eos> && GEOM == kSpherical && NFX <= 0 ? 4 : 0;
    __shared__ double s_sum[kSumLds > 0 ? kSumLds : 1][kSumLds > 0 ? NT : 1];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        if (v < kSumLds) s_sum[v][tid] = 0;
        else r_sum[v] = 0;
    }

    // ring cell of this thread (at most one: NRING <= NT), fixed for the whole march
    static_assert(NRING <= NT, "one ring cell per thread");
    // 3D: the ring is the first wave's work (a scalar branch); 2D: of the wave's first two lanes
    bool const has_ring = ND == 3 && NRING == 64 ? __builtin_amdgcn_readfirstlane(tid) < NRING : tid < NRING;
    int ring_px = 0, ring_py = 0;
    if constexpr (ND == 2) {
        ring_px = tid == 0 ? 0 : PX - 1;
    } else if constexpr (ND == 3) {
        int const r = tid;
        if (r < PX - 2) { ring_px = 1 + r; ring_py = 0; }
        else if (r < 2 * (PX - 2)) { ring_px = 1 + r - (PX - 2); ring_py = PY - 1; }
        else if (r < 2 * (PX - 2) + (PY - 2)) { ring_px = 0; ring_py = 1 + r - 2 * (PX - 2); }
        else { ring_px = PX - 1; ring_py = 1 + r - 2 * (PX - 2) - (PY - 2); }
    }
    int const ring_a = ND >= 2 ? min(ox - 2 + ring_px, G.nwg[0] - 1) : 0;
    int const ring_b = ND == 3 ? min(oy - 2 + ring_py, G.nwg[1] - 1) : 0;

    // pipeline registers.  Global loads run one plane ahead of their use (own column: plane h+2
    // while plane h is processed; ring cell: plane h+1), so their latency hides behind a plane
    // of arithmetic instead of stalling the workgroup at the LDS barrier.  In 3D they are issued
    // after the predictor (kLate), whose face states need the registers more: the Riemann solves
    // still cover the latency (RT 256^3 10.9 -> 11.3 Gcell/s, FP32 21.5 -> 22.0, Sedov 7.4 -> 7.6).
    constexpr bool kLate = ND == 3;
    State<ND, T> pm, p0, pp, c0, cp, cnext, rnext;
    // Carried from plane to plane: the internal energies of c0 and cp that their pressure recovery
    // forms, and dt / dV of plane h-1 for its completion.  The 3D spherical kernels recompute them
    // instead: there the extra registers spill (FP64 Sedov 7.0 -> 7.4 Gcell/s without, FP32 12.6 -> 13.1).
    constexpr bool kCarry = !(ND == 3 && GEOM == kSpherical);
    double e0 = 1, ep = 1;
    T dtodv_prev = 0;
    State<ND, T> fsR_prev, Fm_prev, part_prev;  // in registers, or in s_park when kPark
    T old_rho_prev = 0, old_mom_prev = 0, src_prev = 0;
    // pressure fix: the cell of plane h-1 is rewritten by k_pressure_fix_fused, which also supplies its rate
    bool pf_prev = false, pf_cur = false;
    // set when the fix rewrites some consumed cell of this workgroup (in LDS, not in a register
    // live across the march)
    __shared__ int s_pf_any;
    if (tid == 0) s_pf_any = 0;
    __syncthreads();
    // passive scalars: mass fractions of planes h-1, h, h+1 and the prefetch; the ring cell's
    // prefetch; the right march face of plane h-1, its partial-density update and the
    // upwinded scalar flux of its left march face (godunov_scheme.hpp:263-290)
    X xm = zero_frac<NFX, T>(), x0 = xm, xp = xm, xnext = xm, rxnext = xm;
    X xfR_prev = xm, xpart_prev = xm, ffm_prev = xm;
    int const zfirst = seg_ok ? zs - 1 : 0;
    int const zlast = seg_ok ? ze : -1;
    if (seg_ok) {
        pm = cons_to_prim(load_cons<ND>(A, G, cell_at<ND>(G, a, bb, zfirst - 1)), eos);
        c0 = load_cons<ND>(A, G, cell_at<ND>(G, a, bb, zfirst));
        if constexpr (kCarry) p0 = cons_to_prim_e(c0, eos, e0);
        else p0 = cons_to_prim(c0, eos);
        cnext = load_cons<ND>(A, G, cell_at<ND>(G, a, bb, zfirst + 1));
        if constexpr (NFX > 0) {
            xm = load_frac<NFX>(A, G, cell_at<ND>(G, a, bb, zfirst - 1));
            x0 = load_frac<NFX>(A, G, cell_at<ND>(G, a, bb, zfirst));
            xnext = load_frac<NFX>(A, G, cell_at<ND>(G, a, bb, zfirst + 1));
        }
    }
    if constexpr (ND >= 2) {
        if (has_ring) {
            rnext = load_cons<ND>(A, G, cell_at<ND>(G, ring_a, ring_b, zfirst));
            if constexpr (NFX > 0) rxnext = load_frac<NFX>(A, G, cell_at<ND>(G, ring_a, ring_b, zfirst));
        }
    }

    if constexpr (kPark) {  // plane zfirst-1's primitives of the own column, where the loop reads them
#pragma unroll
        for (int v = 0; v < NV; ++v) s_prim[(zfirst - 1) & 1][v][(ND == 3) ? hy + 1 : 0][hx + 1] = pm[v];
    }
    auto park = [&](int slot, T v) {
        if constexpr (kPark) s_park[slot][tid] = v;
    };
    auto unpark = [&](int slot) -> T {
        if constexpr (kPark) return s_park[slot][tid];
        else return T(0);
    };

    auto prefetch_column = [&](int h) {
        if (h < zlast) {
            cnext = load_cons<ND>(A, G, cell_at<ND>(G, a, bb, h + 2));
            if constexpr (NFX > 0) xnext = load_frac<NFX>(A, G, cell_at<ND>(G, a, bb, h + 2));
        }
    };
    auto prefetch_ring = [&](int h) {
        if (h < zlast) {
            rnext = load_cons<ND>(A, G, cell_at<ND>(G, ring_a, ring_b, h + 1));
            if constexpr (NFX > 0) rxnext = load_frac<NFX>(A, G, cell_at<ND>(G, ring_a, ring_b, h + 1));
        }
    };

    for (int h = zfirst; h <= zlast; ++h) {
        int const pb = h & 1;
        // ---- plane h+1 of this column (prefetched), and the prefetch of plane h+2
        cp = cnext;
        xp = xnext;
        if constexpr (!kLate) prefetch_column(h);
        if constexpr (kCarry) pp = cons_to_prim_e(cp, eos, ep);
        else pp = cons_to_prim(cp, eos);
        // ---- plane h primitives in LDS (own column + ring)
        if constexpr (ND >= 2) {
            // buffer h & 1 was last read at plane h - 2, before the barrier of plane h - 1
#pragma unroll
            for (int v = 0; v < NV; ++v) s_prim[pb][v][(ND == 3) ? hy + 1 : 0][hx + 1] = p0[v];
#pragma unroll
            for (int f = 0; f < NFX; ++f) s_prim[pb][NV + f][(ND == 3) ? hy + 1 : 0][hx + 1] = x0.f[f];
            if (has_ring) {
                State<ND, T> const pr = cons_to_prim(rnext, eos);
#pragma unroll
                for (int v = 0; v < NV; ++v) s_prim[pb][v][ring_py][ring_px] = pr[v];
#pragma unroll
                for (int f = 0; f < NFX; ++f) s_prim[pb][NV + f][ring_py][ring_px] = rxnext.f[f];
                if constexpr (!kLate) prefetch_ring(h);
            }
            __syncthreads();
        }
        int ci, cj, ck;
        ijk_of<ND>(a, bb, h, ci, cj, ck);
        bool const out_plane = h >= zs && h < ze;

        // ---- predictor of plane h
        State<ND, T> fs[2][ND];
        X xf[2][ND];
        double qv = 0;
        if (live) {
            State<ND, T> nb3[ND][2];
            X xnb[ND][2];
            if constexpr (ND >= 2) {
                int const py0 = (ND == 3) ? hy + 1 : 0;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    nb3[0][0][v] = s_prim[pb][v][py0][hx];
                    nb3[0][1][v] = s_prim[pb][v][py0][hx + 2];
                }
#pragma unroll
                for (int f = 0; f < NFX; ++f) {
                    xnb[0][0].f[f] = s_prim[pb][NV + f][py0][hx];
                    xnb[0][1].f[f] = s_prim[pb][NV + f][py0][hx + 2];
                }
                if constexpr (ND == 3) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        nb3[1][0][v] = s_prim[pb][v][hy][hx + 1];
                        nb3[1][1][v] = s_prim[pb][v][hy + 2][hx + 1];
                    }
#pragma unroll
                    for (int f = 0; f < NFX; ++f) {
                        xnb[1][0].f[f] = s_prim[pb][NV + f][hy][hx + 1];
                        xnb[1][1].f[f] = s_prim[pb][NV + f][hy + 2][hx + 1];
                    }
                }
            }
            if constexpr (kPark) {  // plane h-1 of the own column, still in the other buffer
#pragma unroll
                for (int v = 0; v < NV; ++v) nb3[MD][0][v] = s_prim[pb ^ 1][v][(ND == 3) ? hy + 1 : 0][hx + 1];
            } else {
                nb3[MD][0] = pm;
            }
            nb3[MD][1] = pp;
            xnb[MD][0] = xm;
            xnb[MD][1] = xp;
            // dt / dV once per cell where registers allow (kCarry): the half step's (dt / 2) / dV is
            // exactly half of it (a power-of-two scaling commutes with rounding in the normal range)
            T dtodv_h;
            if constexpr (kCarry) {
                qv = fdiv(dt_d, cell_volume<ND, GEOM>(G, ci, cj, ck));
                dtodv_h = T(qv * 0.5);
            } else {
                dtodv_h = T(fdiv(dth_d, cell_volume<ND, GEOM>(G, ci, cj, ck)));
            }
            predict_faces<Eos, ND, GEOM, LIM, NFX>(G, eos, dth, dtodv_h, ci, cj, ck, p0, nb3, fs, x0, xnb, xf);
        } else {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    fs[s][d] = p0;
                    xf[s][d] = x0;
                }
        }

        if constexpr (kLate) {
            prefetch_column(h);
            if (has_ring) prefetch_ring(h);
        }
        // ---- in-plane fluxes and the in-plane part of the update of plane h
        State<ND, T> part = c0;
        T old_rho = c0[0], old_mom = c0[1 + MD], src_m = 0;
        X xpart;  // partial densities fx * rho (godunov_scheme.hpp:122) plus the in-plane fluxes
#pragma unroll
        for (int f = 0; f < NFX; ++f) xpart.f[f] = x0.f[f] * c0[0];
        T dtodv = 0;
        if (out_plane && live) {
            dtodv = kCarry ? T(qv) : T(fdiv(dt_d, cell_volume<ND, GEOM>(G, ci, cj, ck)));
            if (out_col) {
                // min internal energy of the consumed state (internal_energy.cpp:25-40), as its
                // pressure recovery formed it
                r_emin = reduce_combine<kMin>(r_emin, kCarry ? e0 : state_eint<ND>(eos, c0));
                if constexpr (std::is_same_v<Eos, PerfectGas>) {
                    if (A.pf) {
                        pf_cur = pressure_fix_applies(c0, A.eps_pf);  // pressure_fix.hpp:61-68
                        if (pf_cur) s_pf_any = 1;
                    }
                }
            }
        }
        if (out_plane) {
            if constexpr (ND >= 2) {
                // Riemann solve of the left face along in-plane dim p, given the right face state
                // (and scalar face values) of the column on the left; pl and pr are the primitives
                // of its two sides
                auto solve = [&](int p, const State<ND, T>& left, const X& xleft, State<ND, T>& F, X& XF, State<ND, T>& pl, State<ND, T>& pr) {
                    FaceSide<ND, Eos> const L = face_side(left, eos), R = face_side(fs[0][p], eos);
                    F = riemann<RS>(left, fs[0][p], L, R, p, eos);
                    pl = L.p;
                    pr = R.p;
                    // upwind face of the scalar (godunov_scheme.hpp:265-287): this cell's
                    // left face when the mass flux is negative, else the left cell's right face
#pragma unroll
                    for (int f = 0; f < NFX; ++f) XF.f[f] = (F[0] < 0 ? xf[0][p].f[f] : xleft.f[f]) * F[0];
                };
                // the update of dim p (flux, sources, gravity) in the reference order: dims in turn
                auto accumulate = [&](int p, const State<ND, T>& FL, const State<ND, T>& FR, const X& XL, const X& XR, const State<ND, T>& qL,
                                      const State<ND, T>& qR) {
                    T const dS = T(face_area<ND, GEOM>(G, p, ci, cj, ck));
                    T const dSp = T(face_area<ND, GEOM>(G, p, ci + (p == 0), cj + (p == 1), ck));
#pragma unroll
                    for (int v = 0; v < NV; ++v) part[v] += dtodv * ((FL[v] * dS) - (FR[v] * dSp));
                    godunov_sources<Eos, ND, GEOM>(G, p, ci, cj, dtodv, dS, dSp, qL, qR, part);
                    if (gravity_acts(G, p)) {
                        T const g = T(gravity(G, ci, p));
                        part[1 + p] += dt * g * c0[0];
                        part[ND + 1] += dt * g * c0[1 + p];
                    }
#pragma unroll
                    for (int f = 0; f < NFX; ++f) xpart.f[f] += dtodv * ((XL.f[f] * dS) - (XR.f[f] * dSp));
                };
                if (live) {
                    // y (3D): right face states through LDS, in the columns' own slots of the other
                    // primitive plane, whose values (plane h - 1) were last read before this point:
                    // by other columns at plane h - 1, by this one (kPark) above
                    if constexpr (ND == 3) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) s_prim[pb ^ 1][v][hy + 1][hx + 1] = fs[1][1][v];
#pragma unroll
                        for (int f = 0; f < NFX; ++f) s_prim[pb ^ 1][NV + f][hy + 1][hx + 1] = xf[1][1].f[f];
                    }
                    // x: the column at x - 1 is the lane beside
                    State<ND, T> left, FL, FR, pl, qL, qR;
                    X xleft, XL, XR;
#pragma unroll
                    for (int v = 0; v < NV; ++v) left[v] = lane_shift<HX, true>(fs[1][0][v]);
#pragma unroll
                    for (int f = 0; f < NFX; ++f) xleft.f[f] = lane_shift<HX, true>(xf[1][0].f[f]);
                    solve(0, left, xleft, FL, XL, pl, qL);
                    if constexpr (NFX == kStoreMass) {
                        if (x_face) A.mflux[cell_at<ND>(G, a, bb, h)] = FL[0];
                    }
                    // the right face's flux is the left flux of the column at x + 1
#pragma unroll
                    for (int v = 0; v < NV; ++v) FR[v] = lane_shift<HX, false>(FL[v]);
#pragma unroll
                    for (int f = 0; f < NFX; ++f) XR.f[f] = lane_shift<HX, false>(XL.f[f]);
                    if constexpr (GEOM == kSpherical) {  // the primitives of this column's own right face
                        qR[0] = fs[1][0][0];
#pragma unroll
                        for (int v = 1; v < NV; ++v) qR[v] = lane_shift<HX, false>(pl[v]);
                    }
                    accumulate(0, FL, FR, XL, XR, qL, qR);
                }
                if constexpr (ND == 3) {  // y: left states and right fluxes through LDS
                    __syncthreads();
                    State<ND, T> left, FL, FR, pl, qL, qR;
                    X xleft, XL, XR;
                    if (live) {
                        int const hyl = max(hy - 1, 0);
#pragma unroll
                        for (int v = 0; v < NV; ++v) left[v] = s_prim[pb ^ 1][v][hyl + 1][hx + 1];
#pragma unroll
                        for (int f = 0; f < NFX; ++f) xleft.f[f] = s_prim[pb ^ 1][NV + f][hyl + 1][hx + 1];
                        solve(1, left, xleft, FL, XL, pl, qL);
                        if constexpr (NFX == kStoreMass) {
                            if (y_face) A.mflux[cell_at<ND>(G, a, bb, h) + G.plane] = FL[0];
                        }
                        // s_fl was last read before the primitive barrier of this plane
#pragma unroll
                        for (int v = 0; v < NV; ++v) s_fl[v][hy][hx] = FL[v];
#pragma unroll
                        for (int f = 0; f < NFX; ++f) s_fl[NV + f][hy][hx] = XL.f[f];
                        if constexpr (kFaceP) {
#pragma unroll
                            for (int v = 2; v < NV; ++v) s_fp[v - 2][hy][hx] = pl[v];
                        }
                    }
                    __syncthreads();
                    if (live) {
                        int const hyr = min(hy + 1, HY - 1);
#pragma unroll
                        for (int v = 0; v < NV; ++v) FR[v] = s_fl[v][hyr][hx];
#pragma unroll
                        for (int f = 0; f < NFX; ++f) XR.f[f] = s_fl[NV + f][hyr][hx];
                        if constexpr (kFaceP) {
                            qR[0] = fs[1][1][0];
#pragma unroll
                            for (int v = 2; v < NV; ++v) qR[v] = s_fp[v - 2][hyr][hx];
                        }
                        accumulate(1, FL, FR, XL, XR, qL, qR);
                    }
                }
            }
            // geometric pressure source of the march dim (1D spherical: r; 2D spherical: theta)
            if constexpr (GEOM == kSpherical && MD <= 1) {
                if (live) {
                    State<ND, T> const pL = cons_to_prim(fs[0][MD], eos);
                    State<ND, T> const pR = cons_to_prim(fs[1][MD], eos);
                    T const dS = T(face_area<ND, GEOM>(G, MD, ci, cj, ck));
                    T const dSp = T(face_area<ND, GEOM>(G, MD, ci + (MD == 0), cj + (MD == 1), ck));
                    src_m = src_pressure<Eos>(dtodv, pL[ND + 1], pR[ND + 1], dS, dSp);
                }
            }
        }

        // ---- march-dim face h-1/2 and completion of plane h-1
        if (h >= zs && live) {
            if constexpr (kPark) {
#pragma unroll
                for (int v = 0; v < NV; ++v) fsR_prev[v] = unpark(v);
            }
            State<ND, T> const Fm = riemann<RS>(fsR_prev, fs[0][MD], MD, eos);
            if constexpr (NFX == kStoreMass) {  // the face above the last plane belongs to the next segment, or is the last one
                if (out_col && (h < ze || h == G.ngh[MD] + G.n[MD])) A.mflux[cell_at<ND>(G, a, bb, h) + G.plane * MD] = Fm[0];
            }
            X XFm;  // upwinded scalar flux of the face h-1/2
#pragma unroll
            for (int f = 0; f < NFX; ++f) {
                T const xr = kPark ? unpark(3 * NV + f) : xfR_prev.f[f];
                XFm.f[f] = (Fm[0] < 0 ? xf[0][MD].f[f] : xr) * Fm[0];
            }
            int const hm = h - 1;
            if (hm >= zs) {
                int pi, pj, pk;
                ijk_of<ND>(a, bb, hm, pi, pj, pk);
                double const vol = cell_volume<ND, GEOM>(G, pi, pj, pk);
                T const dtodv_m = kCarry ? dtodv_prev : T(fdiv(dt_d, vol));
                T const dS = T(face_area<ND, GEOM>(G, MD, pi, pj, pk));
                T const dSp = T(face_area<ND, GEOM>(G, MD, ci, cj, ck));
                if constexpr (kPark) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        part_prev[v] = unpark(NV + v);
                        Fm_prev[v] = unpark(2 * NV + v);
                    }
#pragma unroll
                    for (int f = 0; f < NFX; ++f) {
                        xpart_prev.f[f] = unpark(3 * NV + NFX + f);
                        ffm_prev.f[f] = unpark(3 * NV + 2 * NFX + f);
                    }
                }
                State<ND, T> un = part_prev;
#pragma unroll
                for (int v = 0; v < NV; ++v) un[v] += dtodv_m * ((Fm_prev[v] * dS) - (Fm[v] * dSp));
                if constexpr (GEOM == kSpherical && MD <= 1) un[1 + MD] += src_prev;
                if (gravity_acts(G, MD)) {
                    T const g = T(gravity(G, pi, MD));
                    un[1 + MD] += dt * g * old_rho_prev;
                    un[ND + 1] += dt * g * old_mom_prev;
                }
                if (out_col) {
                    store_cons<ND>(A, G, cell_at<ND>(G, a, bb, hm), un);
                    if constexpr (NFX > 0) {  // godunov_scheme.hpp:288, then passive_scalar_Godunov (:294-301)
                        int64_t const id = cell_at<ND>(G, a, bb, hm);
#pragma unroll
                        for (int f = 0; f < NFX; ++f) {
                            T const xn = xpart_prev.f[f] + dtodv_m * ((ffm_prev.f[f] * dS) - (XFm.f[f] * dSp));
                            T const y = Eos::div(xn, un[0]);
                            A.fx_new[id + G.plane * f] = y < T(0) ? T(0) : (y > T(1) ? T(1) : y);
                        }
                    }
                    // epilogue: CFL rate of the new state and the conserved totals (FP64); a cell the
                    // pressure fix rewrites gets its rate from k_pressure_fix_fused
                    if (!pf_prev) r_inv = reduce_combine<kMax>(r_inv, state_rate<ND, GEOM>(G, eos, pi, pj, pk, un));
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        if (v < kSumLds) s_sum[v][tid] += (double)un[v] * vol;
                        else r_sum[v] += (double)un[v] * vol;
                    }
                }
            }
            if constexpr (kPark) {
#pragma unroll
                for (int v = 0; v < NV; ++v) park(2 * NV + v, Fm[v]);
#pragma unroll
                for (int f = 0; f < NFX; ++f) park(3 * NV + 2 * NFX + f, XFm.f[f]);
            } else {
                Fm_prev = Fm;
                ffm_prev = XFm;
            }
        }

        // ---- rotate the pipeline
        if constexpr (kPark) {
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                park(v, fs[1][MD][v]);
                park(NV + v, part[v]);
            }
#pragma unroll
            for (int f = 0; f < NFX; ++f) {
                park(3 * NV + f, xf[1][MD].f[f]);
                park(3 * NV + NFX + f, xpart.f[f]);
            }
        } else {
            fsR_prev = fs[1][MD];
            part_prev = part;
            xfR_prev = xf[1][MD];
            xpart_prev = xpart;
        }
        xm = x0;
        x0 = xp;
        old_rho_prev = old_rho;
        old_mom_prev = old_mom;
        src_prev = src_m;
        pf_prev = pf_cur;
        pf_cur = false;
        pm = p0;
        p0 = pp;
        c0 = cp;
        if constexpr (kCarry) {
            e0 = ep;
            dtodv_prev = dtodv;
        }
    }

    // ---- workgroup partials
    r_inv = block_reduce<kMax>(r_inv, s_red, tid, NT);
    r_emin = block_reduce<kMin>(r_emin, s_red, tid, NT);
#pragma unroll
    for (int v = 0; v < NV; ++v) r_sum[v] = block_reduce<kSum>(v < kSumLds ? s_sum[v < kSumLds ? v : 0][tid] : r_sum[v], s_red, tid, NT);
    static_assert(2 + NV < kPartialStride, "the pressure-fix flag has a slot of its own");
    if (tid == 0) {
        double* out = A.partials + (int64_t)blockIdx.x * kPartialStride;
        out[0] = r_inv;
        out[1] = r_emin;
#pragma unroll
        for (int v = 0; v < NV; ++v) out[2 + v] = r_sum[v];
        out[kPartialStride - 1] = s_pf_any ? 1.0 : 0.0;  // the reductions' barriers ordered every write
    }
}

// Runtime dispatch over dimension, geometry, Riemann solver and limiter: calls
// v.template run<ND, GEOM, RS, LIM>() for the configuration given.
template <class V>
static void march_visit(int nd, int geom, int rs, int lim, V&& v)
{
#define HCLPP_F4(NDV, GV, RSV, LV) v.template run<NDV, GV, RSV, LV>()
#define HCLPP_FL(NDV, GV, RSV)                                     \
    switch (lim) {                                                 \
    case kConstant: HCLPP_F4(NDV, GV, RSV, kConstant); break;      \
    case kVanLeer: HCLPP_F4(NDV, GV, RSV, kVanLeer); break;        \
    case kMinmod: HCLPP_F4(NDV, GV, RSV, kMinmod); break;          \
    default: HCLPP_F4(NDV, GV, RSV, kVanAlbada); break;            \
    }
#define HCLPP_FR(NDV, GV)                              \
    switch (rs) {                                      \
    case kHLL: HCLPP_FL(NDV, GV, kHLL); break;         \
    case kHLLC: HCLPP_FL(NDV, GV, kHLLC); break;       \
    default: HCLPP_FL(NDV, GV, kLowMach); break;       \
    }
#define HCLPP_FG(NDV)                                                  \
    if (geom == kSpherical) { HCLPP_FR(NDV, kSpherical); }             \
    else { HCLPP_FR(NDV, kCartesian); }
    switch (nd) {
    case 1: HCLPP_FG(1); break;
    case 2: HCLPP_FG(2); break;
    default: HCLPP_FG(3); break;
    }
#undef HCLPP_F4
#undef HCLPP_FL
#undef HCLPP_FR
#undef HCLPP_FG
}

// Whether a march kernel is built in the tall shape too: 3D with FP64 state (FP32 storage loses its
// third wave per SIMD there: 256^3 12.5 -> 14.7 ms), without a carried scalar.
template <class Eos, int ND, int NFX>
constexpr bool kTallShape = ND == 3 && kFp64State<Eos> && NFX <= 0;

// Launch of k_step_march with the context's plan (shape, tile counts, segment length, workgroups).
template <class Eos, int NFX>
struct MarchLaunch {
    const GridDev& G;
    const MarchPlan& P;
    const Eos& eos;
    const StepArraysT<typename Eos::real>& A;
    hipStream_t s;
    template <int ND, int GEOM, int RS, int LIM, bool TALL>
    void launch() const
    {
        using S = MarchShape<ND, TALL>;
        hipLaunchKernelGGL((k_step_march<Eos, ND, GEOM, RS, LIM, NFX, S::HX, S::HY, S::NT>), dim3((unsigned)P.nb), dim3(S::NT), 0, s, G, eos,
                           A, P.L);
    }
    template <int ND, int GEOM, int RS, int LIM>
    void run() const
    {
        if (P.nb == 0) return;
        if constexpr (kTallShape<Eos, ND, NFX>) {
            if (P.tall) return launch<ND, GEOM, RS, LIM, true>();
        }
        launch<ND, GEOM, RS, LIM, false>();
    }
};

// Resident workgroups per CU of a kernel of nt threads (its registers and LDS decide).
template <class K>
static int resident(K kernel, int nt)
{
    int n = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, nt, 0) == hipSuccess ? n : 0;
}

template <class Eos, int NFX>
struct MarchOccupancy {
    Residency* out;
    template <int ND, int GEOM, int RS, int LIM>
    void run() const
    {
        using S = MarchShape<ND>;
        out->normal = resident(k_step_march<Eos, ND, GEOM, RS, LIM, NFX, S::HX, S::HY, S::NT>, S::NT);
        out->tall = 0;
        if constexpr (kTallShape<Eos, ND, NFX>) {
            using T = MarchShape<ND, true>;
            out->tall = resident(k_step_march<Eos, ND, GEOM, RS, LIM, NFX, T::HX, T::HY, T::NT>, T::NT);
        }
    }
};

}  // namespace hclpp
