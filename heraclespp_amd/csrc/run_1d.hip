// run_1d.hip -- launchers of the multi-step 1D kernel (run_1d.hpp).
#include <hip/hip_runtime.h>

#include "run_1d.hpp"

namespace hclpp {

bool run_1d_fits(int nd, const GridDev& G) { return nd == 1 && G.n[0] <= kRun1dCells && G.ngh[0] >= 2 && G.ngh[0] <= kRun1dGhosts; }

namespace {

template <class Eos, int GEOM, int RS, int LIM>
void launch_one(const GridDev& G, const Eos& eos, const BcSpec& bc, DevClock* clock, int nsteps, const StateBuffers<typename Eos::real>& a,
                const StateBuffers<typename Eos::real>& b, hipStream_t s)
{
    if (G.n[0] + 2 <= kRun1dThreads)
        hipLaunchKernelGGL((k_run_1d<Eos, GEOM, RS, LIM, 1>), dim3(1), dim3(kRun1dThreads), 0, s, G, eos, bc, clock, nsteps, a, b);
    else
        hipLaunchKernelGGL((k_run_1d<Eos, GEOM, RS, LIM, 2>), dim3(1), dim3(kRun1dThreads), 0, s, G, eos, bc, clock, nsteps, a, b);
}

template <class Eos, class... Args>
void launch_any(int geom, int rs, int lim, Args&&... args)
{
#define HCLPP_RL(GV, RSV)                                                          \
    switch (lim) {                                                                 \
    case kConstant: launch_one<Eos, GV, RSV, kConstant>(args...); break;           \
    case kVanLeer: launch_one<Eos, GV, RSV, kVanLeer>(args...); break;             \
    case kMinmod: launch_one<Eos, GV, RSV, kMinmod>(args...); break;               \
    default: launch_one<Eos, GV, RSV, kVanAlbada>(args...); break;                 \
    }
#define HCLPP_RR(GV)                                    \
    switch (rs) {                                       \
    case kHLL: HCLPP_RL(GV, kHLL); break;               \
    case kHLLC: HCLPP_RL(GV, kHLLC); break;             \
    default: HCLPP_RL(GV, kLowMach); break;             \
    }
    if (geom == kSpherical) { HCLPP_RR(kSpherical); }
    else { HCLPP_RR(kCartesian); }
#undef HCLPP_RL
#undef HCLPP_RR
}

}  // namespace

void launch_run_1d(int geom, int rs, int lim, const GridDev& G, const PerfectGas& eos, const BcSpec& bc, DevClock* clock, int nsteps,
                   const StateBuffers<double>& a, const StateBuffers<double>& b, hipStream_t s)
{
    launch_any<PerfectGas>(geom, rs, lim, G, eos, bc, clock, nsteps, a, b, s);
}

void launch_run_1d(int geom, int rs, int lim, const GridDev& G, const PerfectGasMixed& eos, const BcSpec& bc, DevClock* clock, int nsteps,
                   const StateBuffers<float>& a, const StateBuffers<float>& b, hipStream_t s)
{
    launch_any<PerfectGasMixed>(geom, rs, lim, G, eos, bc, clock, nsteps, a, b, s);
}

}  // namespace hclpp
