// Launches of the small-mesh stage kernel (dg_stage_wide.hpp) of one
// polynomial degree.  Included by wide_m{3,4,5}.hip only, each of which
// instantiates launch_wide for its degree.
#pragma once

#include "dg_stage_wide.hpp"
#include "stage_launch.hpp"

namespace nemo_host {

template <int M, typename Real>
int launch_wide(Solver& s, const nemo::StageArgs<M, Real>& a, bool net) {
    constexpr int BE = Tile<M>::BE;
    const dim3 grid{unsigned((s.nelem + BE - 1) / BE)}, block{nemo::WIDE_NT};
    const int eq = s.cfg.equations, vol = s.cfg.volume, surf = s.cfg.surface;
#define NEMO_CASE(E_, V_, S_, K_)                                                                              \
    if (eq == E_ && vol == V_ && surf == S_) {                                                                 \
        hipLaunchKernelGGL((nemo::stage_kernel_wide<E_, M, BE, V_, S_, Real, K_>), grid, block, 0, s.stream, a); \
        return NEMO_OK;                                                                                        \
    }
    if (s.cfg.indicator == NEMO_IND_MLP) {
        if constexpr (M == 4) {
            if (net) {
                NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_HLLC, nemo::IK_MLP)
                NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_RUSANOV, nemo::IK_MLP)
            } else {
                NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_HLLC, nemo::IK_STORED)
                NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_RUSANOV, nemo::IK_STORED)
            }
        }
        return fail(NEMO_ERR_ARG, "the learned indicator is built for the EC volume flux with HLLC or Rusanov");
    }
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_WEAK, nemo::SURF_RUSANOV, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_WEAK, nemo::SURF_HLLC, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_CENTRAL, nemo::SURF_RUSANOV, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_CENTRAL, nemo::SURF_HLLC, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_RUSANOV, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_EULER, nemo::VOL_EC, nemo::SURF_HLLC, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_MHD, nemo::VOL_CENTRAL, nemo::SURF_RUSANOV, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_MHD, nemo::VOL_CENTRAL, nemo::SURF_HLLD, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_MHD, nemo::VOL_EC, nemo::SURF_RUSANOV, nemo::IK_RUNTIME)
    NEMO_CASE(nemo::EQ_MHD, nemo::VOL_EC, nemo::SURF_HLLD, nemo::IK_RUNTIME)
#undef NEMO_CASE
    return fail(NEMO_ERR_ARG, "unsupported equations/volume/surface/n_poly combination");
}

}  // namespace nemo_host
