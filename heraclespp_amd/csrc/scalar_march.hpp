// scalar_march.hpp -- the passive scalars of a fused step, after k_step_march has stored the
// mass flux through every face (StepArraysT::mflux) and the new density.
//
// A scalar needs little of the hydro step: the density and the velocity along each dim
// reconstructed along that dim (for the predictor's mass fluxes and half-step face densities), its
// own slopes, and the Riemann solves' mass fluxes.  So the step runs the hydro kernel once and then
// this one for NF scalars at a time, instead of the whole hydro update once per scalar.  The
// arithmetic is the reference's (extrapolation_reconstruction.hpp:87-88, 105-108, 315-337;
// godunov_scheme.hpp:122, 263-301) on the values the hydro kernel has, so the mass fractions are
// those of the unfused sequence bit for bit.
//
// Tiles, columns and the march are k_step_march's (march_column): one thread per column, a plane at
// a time, plane h's density, in-plane velocities and scalars in LDS with a two-cell ring.  Along x a
// face's upwind value passes between lanes, along y the face values of both sides pass through LDS
// (one barrier for all NF scalars), along the march dim they stay in registers.
// Measured, ten steps with a hydro kernel per scalar / with this kernel: 2D 2048^2 VanLeer two scalars
// 5.6 / 4.1 ms, five 13.0 / 5.9; 3D 250^3 two 49.7 / 25.5, five 119 / 36; spherical 160 x 60 x 60 five
// 7.7 / 3.3.  Bound by FP64 issue (a 3D scalar takes three limited slopes and six divisions).
#pragma once

#include "march.hpp"

namespace hclpp {

// Scalars one launch carries at most: each costs 18 registers and, in 3D, 9 KB of LDS.  Four spill
// some 30 registers in 3D FP64 and still beat two launches of two (250^3 33.1 ms against 34.6, 2D
// 2048^2 4.8 against 5.4, ten steps); five would spill twice that.
constexpr int kScalarGroup = 4;

template <class Eos, int ND, int GEOM, int LIM, int NF, int HX, int HY, int NT>
__global__ __launch_bounds__(NT, ND == 3 ? 2 : 1) void k_scalar_march(GridDev G, StepArraysT<typename Eos::real> A, FusedLayout L)
{
    using T = typename Eos::real;
    using X = Frac<NF, T>;
    constexpr int NP = ND - 1;  // in-plane dims
    constexpr int MD = ND - 1;  // march dim
    constexpr int NQ = ND >= 2 ? 1 + NP : 1;  // density and in-plane velocities in LDS
    constexpr int PX = (ND >= 2) ? HX + 2 : 1;
    constexpr int PY = (ND == 3) ? HY + 2 : 1;
    __shared__ T s_q[2][NQ + NF][PY][PX];
    __shared__ T s_y[2][NF][ND == 3 ? HY : 1][ND == 3 ? HX : 1];  // y face values of both sides

    DevClock const* clk = A.clock;
    if (clk->pub.done || clk->pub.status) return;
    double const dt_d = clk->pub.dt;
    double const dth_d = dt_d / 2;

    int const tid = threadIdx.x;
    MarchColumn const mc = march_column<ND, HX, HY, NT>(G, L, blockIdx.x, gridDim.x, tid);
    int const hx = mc.hx, hy = mc.hy, zs = mc.zs, ze = mc.ze;
    bool const out_col = mc.out_col;
    bool const out_row = ND < 3 || (hy >= 1 && hy <= HY - 2 && mc.bb < G.ngh[1] + G.n[1]);
    // columns beyond the array repeat its last one: valid values, never stored or read by an output
    int const a = ND >= 2 ? min(mc.a, G.nwg[0] - 1) : 0, bb = ND == 3 ? min(mc.bb, G.nwg[1] - 1) : 0;
    int const lx = (ND >= 2) ? hx + 1 : 0, ly = (ND == 3) ? hy + 1 : 0;  // own slot of the LDS planes

    constexpr int NRING = (ND == 3) ? 2 * (PX - 2) + 2 * (PY - 2) : ((ND == 2) ? 2 : 0);
    static_assert(NRING <= NT, "one ring cell per thread");
    bool const has_ring = tid < NRING;
    int ring_px = 0, ring_py = 0;
    if constexpr (ND == 2) {
        ring_px = tid == 0 ? 0 : PX - 1;
    } else if constexpr (ND == 3) {
        if (tid < PX - 2) { ring_px = 1 + tid; ring_py = 0; }
        else if (tid < 2 * (PX - 2)) { ring_px = 1 + tid - (PX - 2); ring_py = PY - 1; }
        else if (tid < 2 * (PX - 2) + (PY - 2)) { ring_px = 0; ring_py = 1 + tid - 2 * (PX - 2); }
        else { ring_px = PX - 1; ring_py = 1 + tid - 2 * (PX - 2) - (PY - 2); }
    }
    int const ring_a = ND >= 2 ? min(mc.ox - 2 + ring_px, G.nwg[0] - 1) : 0;
    int const ring_b = ND == 3 ? min(mc.oy - 2 + ring_py, G.nwg[1] - 1) : 0;

    // density and momenta of a cell or, once divided, its velocities, as the conversion of its state forms them
    struct Q {
        T rho, m[ND];
    };
    auto load_q = [&](int64_t id) {
        Q q;
        q.rho = A.rho[id];
#pragma unroll
        for (int d = 0; d < ND; ++d) q.m[d] = A.rhou[id + G.plane * d];
        return q;
    };
    auto velocity = [&](Q const& c) {
        Q q = c;
#pragma unroll
        for (int d = 0; d < ND; ++d) q.m[d] = Eos::div(c.m[d], c.rho);
        return q;
    };

    int const zfirst = mc.seg_ok ? zs - 1 : 0, zlast = mc.seg_ok ? ze : -1;
    Q qm{}, q0{}, qnext{}, rnext{};
    X xm = zero_frac<NF, T>(), x0 = xm, xnext = xm, rxnext = xm;
    X xfR_prev = xm, xpart_prev = xm, ffm_prev = xm;  // of plane h - 1: right march face, update, left march flux
    T dtodv_prev = 0;
    if (mc.seg_ok) {
        int64_t const id = cell_at<ND>(G, a, bb, zfirst), up = cell_at<ND>(G, a, bb, zfirst + 1) - id;
        qm = velocity(load_q(id - up));
        q0 = velocity(load_q(id));
        qnext = load_q(id + up);
        xm = load_frac<NF>(A, G, id - up);
        x0 = load_frac<NF>(A, G, id);
        xnext = load_frac<NF>(A, G, id + up);
        if (has_ring) {
            int64_t const rid = cell_at<ND>(G, ring_a, ring_b, zfirst);
            rnext = load_q(rid);
            rxnext = load_frac<NF>(A, G, rid);
        }
    }

    for (int h = zfirst; h <= zlast; ++h) {
        int const pb = h & 1;
        int64_t const id = cell_at<ND>(G, a, bb, h), up = cell_at<ND>(G, a, bb, 1) - cell_at<ND>(G, a, bb, 0);
        bool const out_plane = h >= zs && h < ze;
        Q const qp = velocity(qnext);
        X const xp = xnext;
        // ---- plane h in LDS (own column + ring); the barriers are k_step_march's
        if constexpr (ND >= 2) {
            s_q[pb][0][ly][lx] = q0.rho;
#pragma unroll
            for (int d = 0; d < NP; ++d) s_q[pb][1 + d][ly][lx] = q0.m[d];
#pragma unroll
            for (int f = 0; f < NF; ++f) s_q[pb][NQ + f][ly][lx] = x0.f[f];
            if (has_ring) {
                Q const r = velocity(rnext);
                s_q[pb][0][ring_py][ring_px] = r.rho;
#pragma unroll
                for (int d = 0; d < NP; ++d) s_q[pb][1 + d][ring_py][ring_px] = r.m[d];
#pragma unroll
                for (int f = 0; f < NF; ++f) s_q[pb][NQ + f][ring_py][ring_px] = rxnext.f[f];
            }
        }
        // ---- loads of the next plane and of this plane's mass fluxes, ahead of their use
        if (h < zlast) {
            qnext = load_q(id + 2 * up);
            xnext = load_frac<NF>(A, G, id + 2 * up);
            if constexpr (ND >= 2) {
                if (has_ring) {
                    int64_t const rid = cell_at<ND>(G, ring_a, ring_b, h + 1);
                    rnext = load_q(rid);
                    rxnext = load_frac<NF>(A, G, rid);
                }
            }
        }
        T Fx = 0, Fy = 0, Fyp = 0, Fm = 0, rho_new = 1;
        if constexpr (ND >= 2) {  // the face below a column is its own or its left neighbour's
            if (out_plane && out_row && hx >= 1 && mc.a <= G.ngh[0] + G.n[0]) Fx = A.mflux[id];
        }
        if constexpr (ND == 3) {
            if (out_plane && out_col) {
                Fy = A.mflux[id + G.plane];
                Fyp = A.mflux[id + G.plane + G.nwg[0]];
            }
        }
        if (out_col && h >= zs) {
            Fm = A.mflux[id + G.plane * MD];
            if (h > zs) rho_new = A.rho_new[id - up];
        }
        if constexpr (ND >= 2) __syncthreads();

        // ---- predictor: face densities and mass fluxes, their half step, then the scalars'
        int ci, cj, ck;
        ijk_of<ND>(a, bb, h, ci, cj, ck);
        int const idx[3] = {ci, cj, ck};
        double const vol = cell_volume<ND, GEOM>(G, ci, cj, ck);
        T const dtodv_h = T(fdiv(dth_d, vol));
        T const dtodv = T(fdiv(dt_d, vol));
        T dS[ND], dSp[ND], r[2][ND], mass[2][ND], half[2][ND];
        CenterDist hd[ND];
        T dl[ND];
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            hd[d] = center_dist<Eos>(G, d, idx[d]);
            dl[d] = T(G.dx[d][idx[d]]);
            dS[d] = T(face_area<ND, GEOM>(G, d, ci, cj, ck));
            dSp[d] = T(face_area<ND, GEOM>(G, d, ci + (d == 0), cj + (d == 1), ck + (d == 2)));
        }
        // value v of the neighbour at side s (0 below, 1 above) along in-plane dim d
        auto lds = [&](int v, int d, int s) -> T { return s_q[pb][v][ly + (d == 1 ? 2 * s - 1 : 0)][lx + (d == 0 ? 2 * s - 1 : 0)]; };
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            T u[2];
            if (d == MD) {
                reconstruct<LIM, Eos>(qm.rho, q0.rho, qp.rho, hd[d], dl[d], r[0][d], r[1][d]);
                reconstruct<LIM, Eos>(qm.m[d], q0.m[d], qp.m[d], hd[d], dl[d], u[0], u[1]);
            } else {
                reconstruct<LIM, Eos>(lds(0, d, 0), q0.rho, lds(0, d, 1), hd[d], dl[d], r[0][d], r[1][d]);
                reconstruct<LIM, Eos>(lds(NP > 0 ? 1 + d : 0, d, 0), q0.m[d], lds(NP > 0 ? 1 + d : 0, d, 1), hd[d], dl[d], u[0], u[1]);
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) mass[s][d] = r[s][d] * u[s];
        }
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int s = 0; s < 2; ++s) half[s][d] = r[s][d];
#pragma unroll
        for (int e = 0; e < ND; ++e)
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int s = 0; s < 2; ++s) half[s][d] += dtodv_h * ((mass[0][e] * dS[e]) - (mass[1][e] * dSp[e]));
        X xf[2][ND];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            T xo[2][ND];
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                if (d == MD) reconstruct<LIM, Eos>(xm.f[f], x0.f[f], xp.f[f], hd[d], dl[d], xo[0][d], xo[1][d]);
                else reconstruct<LIM, Eos>(lds(NQ + f, d, 0), x0.f[f], lds(NQ + f, d, 1), hd[d], dl[d], xo[0][d], xo[1][d]);
            }
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int s = 0; s < 2; ++s) xf[s][d].f[f] = xo[s][d] * r[s][d];
#pragma unroll
            for (int e = 0; e < ND; ++e) {
                T const inc = dtodv_h * ((xo[0][e] * mass[0][e] * dS[e]) - (xo[1][e] * mass[1][e] * dSp[e]));
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int s = 0; s < 2; ++s) xf[s][d].f[f] += inc;
            }
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int s = 0; s < 2; ++s) xf[s][d].f[f] = Eos::div(xf[s][d].f[f], half[s][d]);
        }

        // ---- in-plane fluxes and their part of the update
        X xpart;
#pragma unroll
        for (int f = 0; f < NF; ++f) xpart.f[f] = x0.f[f] * q0.rho;
        if constexpr (ND >= 2) {
            if (out_plane) {
                if constexpr (ND == 3) {
                    // s_y was last read at plane h - 1, before this plane's barrier
#pragma unroll
                    for (int f = 0; f < NF; ++f) {
                        s_y[0][f][hy][hx] = xf[0][1].f[f];
                        s_y[1][f][hy][hx] = xf[1][1].f[f];
                    }
                }
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    T const below = lane_shift<HX, true>(xf[1][0].f[f]);
                    T const XL = (Fx < 0 ? xf[0][0].f[f] : below) * Fx;
                    T const XR = lane_shift<HX, false>(XL);
                    xpart.f[f] += dtodv * ((XL * dS[0]) - (XR * dSp[0]));
                }
                if constexpr (ND == 3) {
                    __syncthreads();
                    int const hyl = max(hy - 1, 0), hyr = min(hy + 1, HY - 1);
#pragma unroll
                    for (int f = 0; f < NF; ++f) {
                        T const XL = (Fy < 0 ? xf[0][1].f[f] : s_y[1][f][hyl][hx]) * Fy;
                        T const XR = (Fyp < 0 ? s_y[0][f][hyr][hx] : xf[1][1].f[f]) * Fyp;
                        xpart.f[f] += dtodv * ((XL * dS[1]) - (XR * dSp[1]));
                    }
                }
            }
        }
        // ---- march face h - 1/2 and completion of plane h - 1
        if (h >= zs) {
            X ffm;
#pragma unroll
            for (int f = 0; f < NF; ++f) ffm.f[f] = (Fm < 0 ? xf[0][MD].f[f] : xfR_prev.f[f]) * Fm;
            if (h > zs && out_col) {
                int pi, pj, pk;
                ijk_of<ND>(a, bb, h - 1, pi, pj, pk);
                T const dSm = T(face_area<ND, GEOM>(G, MD, pi, pj, pk));
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    T const xn = xpart_prev.f[f] + dtodv_prev * ((ffm_prev.f[f] * dSm) - (ffm.f[f] * dS[MD]));
                    T const y = Eos::div(xn, rho_new);
                    A.fx_new[id - up + G.plane * f] = y < T(0) ? T(0) : (y > T(1) ? T(1) : y);
                }
            }
            ffm_prev = ffm;
        }
        // ---- rotate the pipeline
#pragma unroll
        for (int f = 0; f < NF; ++f) xfR_prev.f[f] = xf[1][MD].f[f];
        xpart_prev = xpart;
        dtodv_prev = dtodv;
        xm = x0;
        x0 = xp;
        qm = q0;
        q0 = qp;
    }
}

}  // namespace hclpp
