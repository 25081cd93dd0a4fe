// clock.hpp -- the device clock: what main.cpp's loop decides between two steps, by one thread.
#pragma once

#include <hip/hip_runtime.h>

#include "fused.hpp"

namespace hclpp {

// main.cpp:355-385 (dt, output clipping, t_end clip, max_iter) and :397-425 (internal energy check)
__device__ __forceinline__ void schedule_next(DevClock* c, double inv)
{
    double dt = c->pub.cfl * (1 / inv);
    int pending = 0, output = 0;
    if (c->iter_output_frequency > 0) {  // :362-368 (iter_ini = 0)
        int const next_output = (c->pub.iter_output_id + 1) * c->iter_output_frequency;
        if ((c->pub.iter + 1) >= next_output) {
            output = 1;
            c->pub.iter_output_id += 1;
        }
    }
    if (c->time_output_frequency > 0) {  // :369-375
        double const next_output = c->time_first_output + ((c->pub.time_output_id + 1) * c->time_output_frequency);
        if ((c->pub.t + dt) >= next_output) {
            dt = next_output - c->pub.t;
            if (dt <= 0) {
                c->pub.status = HCLPP_ERR_NEGATIVE_DT;
                return;
            }
            output = 1;
            c->pub.time_output_id += 1;
        }
    }
    if ((c->pub.t + dt) >= c->pub.t_end) {
        dt = c->pub.t_end - c->pub.t;
        output = 1;
        pending = 1;
    }
    if ((c->pub.iter + 1) >= c->pub.max_iter) {
        output = 1;
        pending = 1;
    }
    c->pub.dt = dt;
    c->pending_exit = pending;
    c->pending_output = output;
}

// The end of a step: the internal-energy check, the step's time and totals, exits and output pauses,
// then the next dt.  inv: max CFL rate of the new state; emin: min internal energy of the state the
// step read; s: conserved totals of the new state.
template <int NV>
__device__ __forceinline__ void clock_finish(DevClock* c, double inv, double emin, const double (&s)[NV])
{
    c->pub.min_eint = emin;
    if (isnan(emin) || emin < 0) {
        c->pub.status = 3;  // HCLPP_ERR_STATE: the step is discarded
        return;
    }
    if (c->dt_log && c->pub.iter < c->dt_log_cap) c->dt_log[c->pub.iter] = c->pub.dt;
    c->pub.t += c->pub.dt;
    c->pub.iter += 1;
    c->pub.mass = s[0];
#pragma unroll
    for (int d = 0; d < 3; ++d) c->pub.momentum[d] = d < NV - 2 ? s[1 + d] : 0.;
    c->pub.energy = s[NV - 1];
    c->pub.output_due = c->pending_output;
    if (c->pending_exit) {
        c->pub.done = 1;
        c->pub.exiting = 1;
        return;
    }
    if (c->pending_output) {  // pause: the caller writes the output, then starts the clock again
        c->pub.done = 1;
        return;
    }
    schedule_next(c, inv);
}

}  // namespace hclpp
