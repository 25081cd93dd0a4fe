// run_1d.hpp -- several fused steps of a small 1D grid in one launch (k_run_1d).
//
// A 1D grid of up to two thousand cells gives a step's three kernels (march, ghost fill, clock) next
// to nothing to do: they are three launches of some microseconds in a row.  One workgroup holds the
// whole state in LDS instead and runs step after step, the clock included, with barriers in place of
// launches.  The per-cell arithmetic is the march kernel's (predict_faces, riemann, state_rate), so
// every conserved value, dt and minimum is the same bit for bit; only the conserved totals are summed
// in another order.  Bound by the serial chain of a step (5 us with 64 cells) and, from some hundred
// cells on, by the FP64 issue of the one CU it occupies.  Measured per step, launch by launch / here: 64
// cells 17 / 5.1 us, 1000 18.3 / 8.1, 2046 18 / 11.2; beyond that two cells per thread no longer fit.
#pragma once

#include "clock.hpp"
#include "march.hpp"

namespace hclpp {

constexpr int kRun1dThreads = 1024;
constexpr int kRun1dGhosts = 4;                        // ghost layers at most
constexpr int kRun1dCells = 2 * kRun1dThreads - 2;     // two faces' cells per thread: n + 2 predictors

// Rate and internal energy of a new state with the primitives the next step starts from
// (state_rate's arithmetic: it forms the same primitives).
template <int GEOM, class Eos>
__device__ __forceinline__ double rate_and_prim(const GridDev& G, const Eos& eos, int i, const State<1, typename Eos::real>& c,
                                                State<1, typename Eos::real>& p, double& e)
{
    double y;
    p = cons_to_prim_ey(c, eos, e, y);
    if constexpr (std::is_same_v<Eos, PerfectGas>) return cfl_rate<1, GEOM>(G, i, 0, 0, &p.q[1], eos.sound(p[0], p[2], y));
    else return state_rate<1, GEOM>(G, eos, i, 0, 0, c);
}

// C: predictor cells per thread.
//
// A step takes three passes over the cells (face states; fluxes; update) with a barrier after each,
// and a fourth barrier for the clock.  The update also forms the primitives, the internal energy and
// the ghosts the next step starts from: the owner of a boundary cell writes the ghosts filled from it.
// The totals, which only the last step leaves in the clock, are summed once at the end.
template <class Eos, int GEOM, int RS, int LIM, int C>
__global__ __launch_bounds__(kRun1dThreads) void k_run_1d(GridDev G, Eos eos, BcSpec bc, DevClock* clock, int nsteps,
                                                          StateBuffers<typename Eos::real> a, StateBuffers<typename Eos::real> b)
{
    using T = typename Eos::real;
    using St = State<1, T>;
    constexpr int NT = kRun1dThreads, NV = 3, NW = NT / 64;
    constexpr int NC = C * NT - 2 + 2 * kRun1dGhosts;
    __shared__ T s_prim[NV][NC];
    __shared__ T s_right[NV][NC];  // right face states
    __shared__ T s_flux[NV][NC];   // fluxes through the faces below the cells; at the end, the state
    __shared__ double s_red[NW][NV];
    __shared__ DevClock s_clk;

    int const tid = threadIdx.x;
    if (clock->pub.done || clock->pub.status) return;
    if (tid == 0) s_clk = *clock;
    int const ng = G.ngh[0], n = G.n[0], ext = G.nwg[0];
    auto get = [](T const (&x)[NV][NC], int i) {
        St q;
#pragma unroll
        for (int v = 0; v < NV; ++v) q[v] = x[v][i];
        return q;
    };
    auto put = [](T (&x)[NV][NC], int i, St const& q) {
#pragma unroll
        for (int v = 0; v < NV; ++v) x[v][i] = q[v];
    };
    auto cell = [&](int c) { return ng - 1 + tid + c * NT; };  // predictor cells ng - 1 .. ng + n
    auto interior = [&](int i) { return i >= ng && i < ng + n; };
    auto load = [&](int i) {
        St q;
        q[0] = a.rho[i];
        q[1] = a.rhou[i];
        q[2] = a.E[i];
        return q;
    };
    // ghost g (0 .. 2 ng - 1, the left ones first): its cell, and the cell it is filled from
    auto ghost_cell = [&](int g) { return g < ng ? g : n + g; };
    auto ghost_source = [&](int g, bool& flip) { return face_map(bc.kind[g < ng ? 0 : 1], ghost_cell(g), ng, n, ext, flip); };

    St cons[C];              // interior cells of this thread
    double emin_next = reduce_identity<kMin>();
    for (int i = tid; i < ext; i += NT) put(s_prim, i, cons_to_prim(load(i), eos));
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (interior(cell(c))) {
            double e;
            cons[c] = load(cell(c));
            cons_to_prim_e(cons[c], eos, e);
            emin_next = reduce_combine<kMin>(emin_next, e);
        }
    __syncthreads();
    Frac<0, T> const no_frac = zero_frac<0, T>();
    int done_steps = 0;
    for (int step = 0; step < nsteps && !s_clk.pub.done && !s_clk.pub.status; ++step) {
        double const dt_d = s_clk.pub.dt;
        int const iter = s_clk.pub.iter;
        double const dth_d = dt_d / 2;
        T const dt = T(dt_d), dth = T(dth_d);
        // ---- face states after the half step
        St left[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            int const i = cell(c);
            if (i > ng + n) break;
            St const nb[1][2] = {{get(s_prim, i - 1), get(s_prim, i + 1)}};
            St fs[2][1];
            Frac<0, T> const xnb[1][2] = {{no_frac, no_frac}};
            Frac<0, T> xf[2][1];
            double const qv = fdiv(dt_d, cell_volume<1, GEOM>(G, i, 0, 0));
            predict_faces<Eos, 1, GEOM, LIM, 0>(G, eos, dth, T(qv * 0.5), i, 0, 0, get(s_prim, i), nb, fs, no_frac, xnb, xf);
            left[c] = fs[0][0];
            put(s_right, i, fs[1][0]);
        }
        __syncthreads();
        // ---- the flux through the face below each cell
#pragma unroll
        for (int c = 0; c < C; ++c) {
            int const i = cell(c);
            if (i >= ng && i <= ng + n) put(s_flux, i, riemann<RS>(get(s_right, i - 1), left[c], 0, eos));
        }
        __syncthreads();
        // ---- update, and the next step's primitives (the predictor has read this step's)
        double inv = reduce_identity<kMax>(), emin = emin_next;
        emin_next = reduce_identity<kMin>();
        St un[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            int const i = cell(c);
            if (!interior(i)) continue;
            un[c] = cons[c];
            T const dtodv = T(fdiv(dt_d, cell_volume<1, GEOM>(G, i, 0, 0)));
            T const dS = T(face_area<1, GEOM>(G, 0, i, 0, 0)), dSp = T(face_area<1, GEOM>(G, 0, i + 1, 0, 0));
#pragma unroll
            for (int v = 0; v < NV; ++v) un[c][v] += dtodv * ((s_flux[v][i] * dS) - (s_flux[v][i + 1] * dSp));
            if constexpr (GEOM == kSpherical) {
                St const pL = cons_to_prim(left[c], eos), pR = cons_to_prim(get(s_right, i), eos);
                un[c][1] += src_pressure<Eos>(dtodv, pL[2], pR[2], dS, dSp);
            }
            if (gravity_acts(G, 0)) {
                T const g = T(gravity(G, i, 0));
                un[c][1] += dt * g * cons[c][0];
                un[c][2] += dt * g * cons[c][1];
            }
            St p;
            double e;
            inv = reduce_combine<kMax>(inv, rate_and_prim<GEOM>(G, eos, i, un[c], p, e));
            emin_next = reduce_combine<kMin>(emin_next, e);
            put(s_prim, i, p);
            if (i < 2 * ng || i >= n) {  // ghosts are filled from the ng cells at either end
                for (int g = 0; g < 2 * ng; ++g) {
                    bool flip = false;
                    if (ghost_source(g, flip) != i) continue;
                    St q = un[c];
                    if (flip) q[1] = -q[1];
                    inv = reduce_combine<kMax>(inv, rate_and_prim<GEOM>(G, eos, ghost_cell(g), q, p, e));
                    put(s_prim, ghost_cell(g), p);
                }
            }
        }
        // ---- reductions and the clock
        inv = wave_reduce<kMax>(inv);
        emin = wave_reduce<kMin>(emin);
        if ((tid & 63) == 0) {
            s_red[tid >> 6][0] = inv;
            s_red[tid >> 6][1] = emin;
        }
        __syncthreads();
        if (tid < 64) {  // the waves' results, by the first wave
            inv = s_red[tid % NW][0];
            emin = s_red[tid % NW][1];
#pragma unroll
            for (int o = NW / 2; o > 0; o >>= 1) {
                inv = reduce_combine<kMax>(inv, __shfl_xor(inv, o, 64));
                emin = reduce_combine<kMin>(emin, __shfl_xor(emin, o, 64));
            }
            if (tid == 0) {
                DevClock k = s_clk;  // in registers: one round of LDS reads, one of writes
                double const totals[NV] = {k.pub.mass, k.pub.momentum[0], k.pub.energy};
                clock_finish<NV>(&k, inv, emin, totals);
                s_clk = k;
            }
        }
        __syncthreads();
        if (s_clk.pub.iter == iter) break;  // the step is discarded: cons is the state it read
#pragma unroll
        for (int c = 0; c < C; ++c) cons[c] = un[c];
        ++done_steps;
    }
    // the state after k steps belongs in the buffer that k alternating steps end in
    if (done_steps > 0) {
        double s[NV] = {0, 0, 0};
#pragma unroll
        for (int c = 0; c < C; ++c) {
            int const i = cell(c);
            if (!interior(i)) continue;
            put(s_flux, i, cons[c]);
            double const vol = cell_volume<1, GEOM>(G, i, 0, 0);
#pragma unroll
            for (int v = 0; v < NV; ++v) s[v] += (double)cons[c][v] * vol;
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            s[v] = wave_reduce<kSum>(s[v]);
            if ((tid & 63) == 0) s_red[tid >> 6][v] = s[v];
        }
        __syncthreads();
        StateBuffers<T> const& out = done_steps % 2 ? b : a;
        for (int i = tid; i < ext; i += NT) {
            bool flip = false;
            St q = get(s_flux, face_map(bc.kind[i < ng ? 0 : 1], i, ng, n, ext, flip));
            if (flip) q[1] = -q[1];
            out.rho[i] = q[0];
            out.rhou[i] = q[1];
            out.E[i] = q[2];
        }
        if (tid == 0) {
            double t[NV] = {0, 0, 0};
            for (int w = 0; w < NW; ++w)
#pragma unroll
                for (int v = 0; v < NV; ++v) t[v] += s_red[w][v];
            s_clk.pub.mass = t[0];
            s_clk.pub.momentum[0] = t[1];
            s_clk.pub.energy = t[2];
        }
    }
    if (tid == 0) *clock = s_clk;
}

}  // namespace hclpp
