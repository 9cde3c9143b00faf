// Which form of the stage kernel a mesh, or a degree group of the ensemble,
// takes: stage_kernel (a block on one wavefront) or the small-mesh form
// stage_kernel_wide (on four).
#pragma once

#include <cstdint>

#include "../../include/nemo_gpu.h"

namespace nemo_host {

// Largest number of blocks for which the small-mesh form is taken: where its
// time per stage crosses that of stage_kernel.  Measured on meshes of 4^3 to
// 32^3 elements (us per stage with a fifth of the step's CFL reduction,
// stage_kernel -> small-mesh form):
//   Euler FP64, EC, HLLC   N = 2:  10 blocks 26.1 -> 12.8, 1143 38.2 -> 34.0, 1739 43.1 -> 43.0, 2812 54.3 -> 62.0
//                          N = 3:  16 33.7 -> 15.1, 1024 38.0 -> 34.1, 1458 50.8 -> 46.4, 2000 49.8 -> 55.5
//                          N = 4:  32 41.2 -> 19.0, 1099 61.2 -> 54.1, 2048 68.3 -> 77.1
//   weak form              N = 3:  16 17.2 -> 10.2, 1024 24.3 -> 22.6, 1458 32.3 -> 33.8
//   Euler FP32, EC, HLLC   N = 2:  10 21.8 -> 11.3, 1739 32.4 -> 28.8, 2812 38.0 -> 38.9
//                          N = 3:  16 25.8 -> 11.8, 1024 28.7 -> 21.8, 4921 72.7 -> 68.6, 8192 97.2 -> 97.4
//             EC, Rusanov  N = 3:  4813 62.0 -> 64.0
//                          N = 4:  32 31.2 -> 13.3, 1099 42.7 -> 33.0, 2048 45.1 -> 46.7
//   GLM-MHD FP64, EC, HLLD N = 2:  10 40.9 -> 18.9, 314 42.7 -> 34.9, 586 42.5 -> 47.8
//                          N = 3:  128 48.7 -> 21.6, 333 47.9 -> 36.5, 550 47.7 -> 51.1
//                          N = 4:  256 76.2 -> 24.9, 2916 293 -> 217, 10976 1133 -> 833
//             EC, Rusanov  N = 4:  256 47.4 -> 21.9, 666 55.2 -> 57.0
//   GLM-MHD FP32, EC, HLLD N = 2:  74 35.9 -> 16.2, 1143 44.4 -> 41.5, 1975 51.0 -> 57.9
//                          N = 3:  128 40.2 -> 17.6, 1458 55.9 -> 49.5, 2000 56.6 -> 57.8
//                          N = 4:  256 57.3 -> 18.2, 2916 229 -> 97.5, 10976 825 -> 364
//             EC, Rusanov  N = 4:  1099 55.0 -> 45.2, 2048 57.4 -> 59.4
// HLLD at N = 4 takes it at any size: there stage_kernel keeps the terms of
// three directions' code in one register allocation and spills 1 to 2 KB per
// lane.
template <int M, typename Real>
long long wide_blocks(const nemo_gpu_config& c) {
    constexpr bool F32 = sizeof(Real) == 4;
    if (c.equations == NEMO_EQ_GLM_MHD) {
        if (M == 5 && c.surface == NEMO_SURF_HLLD) return INT64_MAX;
        if (!F32) return 400;
        return M == 3 ? 1200 : 1536;
    }
    if (!F32) return c.volume == NEMO_VOL_WEAK ? 1024 : (M == 5 ? 1280 : 1536);
    if (M == 4) return c.surface == NEMO_SURF_HLLC ? 6144 : 4096;
    return M == 3 ? 2048 : 1536;
}

// Whether a launch over nblocks blocks takes the small-mesh form; `form` is
// NEMO_FORM_AUTO or one of the two.
template <int M, typename Real>
bool wide_form(const nemo_gpu_config& c, int form, long long nblocks) {
    return form == NEMO_FORM_AUTO ? nblocks <= wide_blocks<M, Real>(c) : form == NEMO_FORM_FOUR_WAVES;
}

}  // namespace nemo_host
