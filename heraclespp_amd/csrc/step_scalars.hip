// step_scalars.hip -- launchers of the passive-scalar kernel (k_scalar_march, scalar_march.hpp).
#include <hip/hip_runtime.h>

#include "scalar_march.hpp"

namespace hclpp {

// Calls v.template run<ND, GEOM, LIM, NF>() for a configuration and a group of nf scalars.
template <class V>
static void scalar_visit(int nd, int geom, int lim, int nf, V&& v)
{
#define HCLPP_SN(NDV, GV, LV)                                      \
    switch (nf) {                                                  \
    case 1: v.template run<NDV, GV, LV, 1>(); break;               \
    case 2: v.template run<NDV, GV, LV, 2>(); break;               \
    case 3: v.template run<NDV, GV, LV, 3>(); break;               \
    default: v.template run<NDV, GV, LV, kScalarGroup>(); break;   \
    }
#define HCLPP_SL(NDV, GV)                          \
    switch (lim) {                                 \
    case kConstant: HCLPP_SN(NDV, GV, kConstant); break; \
    case kVanLeer: HCLPP_SN(NDV, GV, kVanLeer); break;   \
    case kMinmod: HCLPP_SN(NDV, GV, kMinmod); break;     \
    default: HCLPP_SN(NDV, GV, kVanAlbada); break;       \
    }
#define HCLPP_SG(NDV)                                        \
    if (geom == kSpherical) { HCLPP_SL(NDV, kSpherical); }   \
    else { HCLPP_SL(NDV, kCartesian); }
    switch (nd) {
    case 1: HCLPP_SG(1); break;
    case 2: HCLPP_SG(2); break;
    default: HCLPP_SG(3); break;
    }
#undef HCLPP_SN
#undef HCLPP_SL
#undef HCLPP_SG
}

template <class Eos>
struct ScalarLaunch {
    const GridDev& G;
    const MarchPlan& P;
    const StepArraysT<typename Eos::real>& A;
    hipStream_t s;
    template <int ND, int GEOM, int LIM, int NF, bool TALL>
    void launch() const
    {
        using S = MarchShape<ND, TALL>;
        hipLaunchKernelGGL((k_scalar_march<Eos, ND, GEOM, LIM, NF, S::HX, S::HY, S::NT>), dim3((unsigned)P.nb), dim3(S::NT), 0, s, G, A, P.L);
    }
    template <int ND, int GEOM, int LIM, int NF>
    void run() const
    {
        if constexpr (kTallShape<Eos, ND, 0>) {
            if (P.tall) return launch<ND, GEOM, LIM, NF, true>();
        }
        launch<ND, GEOM, LIM, NF, false>();
    }
};

template <class Eos>
struct ScalarOccupancy {
    Residency* out;
    template <int ND, int GEOM, int LIM, int NF>
    void run() const
    {
        using S = MarchShape<ND>;
        out->normal = resident(k_scalar_march<Eos, ND, GEOM, LIM, NF, S::HX, S::HY, S::NT>, S::NT);
        out->tall = 0;
        if constexpr (kTallShape<Eos, ND, 0>) {
            using T = MarchShape<ND, true>;
            out->tall = resident(k_scalar_march<Eos, ND, GEOM, LIM, NF, T::HX, T::HY, T::NT>, T::NT);
        }
    }
};

// As few launches as the group size allows, of nearly equal size (five scalars: 3 + 2).
template <class Eos>
static void launch_scalars_any(int nd, int geom, int lim, const GridDev& G, const MarchPlan& P, const StepArraysT<typename Eos::real>& A, hipStream_t s)
{
    if (P.nb == 0) return;
    int const groups = scalar_groups(A.nfx);
    for (int g = 0, f = 0; g < groups; ++g) {
        int const nf = A.nfx / groups + (g < A.nfx % groups ? 1 : 0);
        StepArraysT<typename Eos::real> Ag = A;
        Ag.fx = A.fx + G.plane * f;
        Ag.fx_new = A.fx_new + G.plane * f;
        Ag.nfx = nf;
        scalar_visit(nd, geom, lim, nf, ScalarLaunch<Eos>{G, P, Ag, s});
        f += nf;
    }
}

int scalar_groups(int nfx) { return (nfx + kScalarGroup - 1) / kScalarGroup; }

void launch_scalar_march(int nd, int geom, int lim, const GridDev& G, const MarchPlan& P, const PerfectGas&, const StepArrays& A, hipStream_t s)
{
    launch_scalars_any<PerfectGas>(nd, geom, lim, G, P, A, s);
}

void launch_scalar_march(int nd, int geom, int lim, const GridDev& G, const MarchPlan& P, const PerfectGasMixed&, const StepArraysF& A, hipStream_t s)
{
    launch_scalars_any<PerfectGasMixed>(nd, geom, lim, G, P, A, s);
}

Residency scalar_occupancy(int nd, int geom, int lim, int nfx, bool fp32)
{
    int const groups = scalar_groups(nfx);
    int const nf = (nfx + groups - 1) / groups;  // the largest group
    Residency n{};
    if (fp32) scalar_visit(nd, geom, lim, nf, ScalarOccupancy<PerfectGasMixed>{&n});
    else scalar_visit(nd, geom, lim, nf, ScalarOccupancy<PerfectGas>{&n});
    return n;
}

}  // namespace hclpp
