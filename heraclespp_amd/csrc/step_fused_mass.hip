// step_fused_mass.hip -- launchers of the fused step (k_step_march, march.hpp) that also stores the
// mass flux through every face, for the passive-scalar kernel that follows it (scalar_march.hpp).
// A translation unit of its own so that its instantiations compile in parallel with the others.
#include <hip/hip_runtime.h>

#include "march.hpp"

namespace hclpp {

void launch_fused_step_mass(int nd, int geom, int rs, int lim, const GridDev& G, const MarchPlan& P, const PerfectGas& eos, const StepArrays& A,
                            hipStream_t s)
{
    march_visit(nd, geom, rs, lim, MarchLaunch<PerfectGas, kStoreMass>{G, P, eos, A, s});
}

void launch_fused_step_mass(int nd, int geom, int rs, int lim, const GridDev& G, const MarchPlan& P, const PerfectGasMixed& eos,
                            const StepArraysF& A, hipStream_t s)
{
    march_visit(nd, geom, rs, lim, MarchLaunch<PerfectGasMixed, kStoreMass>{G, P, eos, A, s});
}

Residency march_occupancy_mass(int nd, int geom, int rs, int lim, bool fp32)
{
    Residency n{};
    if (fp32) march_visit(nd, geom, rs, lim, MarchOccupancy<PerfectGasMixed, kStoreMass>{&n});
    else march_visit(nd, geom, rs, lim, MarchOccupancy<PerfectGas, kStoreMass>{&n});
    return n;
}

}  // namespace hclpp
