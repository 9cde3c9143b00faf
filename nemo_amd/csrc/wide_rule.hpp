// Which form of the stage kernel a mesh, or a degree group of the ensemble,
// takes: stage_kernel (a block on one wavefront) or the small-mesh form
// stage_kernel_wide (on four).
#pragma once

#include <cstdint>

#include "../../include/nemo_gpu.h"

namespace nemo_host {

// Largest number of blocks for which the small-mesh form is taken.  The times
// of both forms are steps: the small-mesh form runs rounds of 512 blocks (two
// workgroups on each of 256 CUs; GLM-MHD in FP64 one), the other of 2048 (of
// 3072 in the FP32 Euler operator), so their curves cross more than once.  A
// limit is the end of the range from one block on in which no measured mesh
// was slower (by more than 1.5 %) than on one wavefront.  What moves it is how
// much of stage_kernel's chain the small-mesh form takes off: the
// Persson-Peraire indicator, which runs beside the other passes there, HLLC,
// the two-point fluxes and the unfused update of SSPRK lengthen the chain; weak
// form and Rusanov alone shorten it.  Up to 512 blocks it is faster in every
// scheme.
//
// Measured with both forms of one build on about 20 meshes of 115 to 6144
// blocks for every entry (us per stage with a fifth of the step's CFL
// reduction, stage_kernel -> small-mesh form, below and above the limit):
//   FP64 N = 2  weak, Rusanov, none, LSRK    483 17.3 -> 13.9    520 16.1 -> 17.9
//               EC, HLLC, none, LSRK         768 23.7 -> 21.4    834 25.5 -> 26.5
//               EC, HLLC, PP, LSRK          1522 39.5 -> 38.1   1536 32.9 -> 36.2
//        N = 3  weak, Rusanov, none, SSPRK  1024 24.8 -> 22.6   1229 30.6 -> 29.9
//               EC, Rusanov, none, LSRK      768 25.9 -> 24.5    844 28.7 -> 29.6
//               EC, HLLC, PP, LSRK          1536 47.3 -> 44.6   2000 49.5 -> 55.5
//        N = 4  central, HLLC, none, LSRK    500 24.1 -> 23.2    520 22.3 -> 28.0
//               EC, HLLC, PP, LSRK          1274 66.9 -> 56.3   1463 60.5 -> 61.8
//   FP32 N = 2  weak, Rusanov, none, LSRK    980 19.7 -> 16.3   1522 23.3 -> 22.5
//               EC, HLLC, PP, LSRK          2048 31.6 -> 31.4   2511 37.5 -> 37.0
//        N = 3  weak, HLLC, none, LSRK      1229 27.4 -> 25.9   2000 29.3 -> 34.2
//               EC, HLLC, none, LSRK        1715 34.2 -> 31.6   2000 32.1 -> 33.0
//               EC, HLLC, PP, LSRK          5103 78.0 -> 73.8   6098 82.8 -> 85.5
//               EC, HLLC, learned, LSRK     1792 37.6 -> 35.9   2560 43.9 -> 45.5
//        N = 4  weak, Rusanov, PP, LSRK     1274 31.6 -> 30.5   1800 31.7 -> 38.6
//               EC, HLLC, PP, LSRK          1536 43.0 -> 36.2   2048 45.7 -> 47.0
// (10 to 256 blocks: 1.3 to 2.9 times faster.)  Weak form and central fluxes
// share an entry, the smaller of their limits.  The learned indicator, whose
// stages 2 to 5 read its factor back, takes the entries without an indicator.
// Meshes beyond a limit may be faster in this form again at the end of a round
// (FP32 N = 3 weak, Rusanov, SSPRK, 2800 blocks: 34.8 -> 35.5, 4200: 55.3 ->
// 48.7); they are left to stage_kernel.  No entry lies above the largest mesh
// measured.
//
// [FP32][n_poly - 2][EC][HLLC][Persson-Peraire][SSPRK]
constexpr int16_t EULER_WIDE[2][3][2][2][2][2] = {
    {{{{{512, 512}, {512, 512}}, {{512, 512}, {1280, 1408}}},
      {{{512, 512}, {1024, 1280}}, {{768, 1280}, {1408, 1536}}}},
     {{{{512, 1024}, {768, 1024}}, {{768, 1280}, {1536, 1536}}},
      {{{768, 1280}, {1280, 1280}}, {{1280, 1536}, {1536, 1536}}}},
     {{{{512, 512}, {512, 512}}, {{512, 512}, {512, 512}}},
      {{{768, 1280}, {1280, 1280}}, {{512, 512}, {1280, 1280}}}}},
    {{{{{1024, 2048}, {2048, 2048}}, {{1664, 2048}, {2048, 2048}}},
      {{{2048, 2048}, {2048, 2048}}, {{1664, 2048}, {2048, 2048}}}},
     {{{{768, 2560}, {1536, 2560}}, {{1280, 1536}, {1536, 2560}}},
      {{{1536, 2560}, {2560, 4096}}, {{1792, 5632}, {5120, 6144}}}},
     {{{{1280, 1536}, {1280, 1536}}, {{1280, 1536}, {1536, 1536}}},
      {{{1280, 1536}, {1536, 1536}}, {{1536, 1536}, {1536, 1536}}}}}};

// GLM-MHD (either indicator and Runge-Kutta scheme), measured as above:
//   FP64  N = 2  EC, Rusanov, none   392 25.6 -> 23.9    622 29.6 -> 37.2
//         N = 3  EC, HLLD, PP        396 43.8 -> 34.7    637 47.6 -> 50.4
//         N = 4  EC, Rusanov, PP     365 51.5 -> 37.0    605 55.7 -> 54.8
//   FP32  N = 2  EC, HLLD, PP       1200 39.4 -> 36.1   1739 46.6 -> 49.4
//                central, Rus., none 980 31.1 -> 27.6   1400 32.6 -> 33.1
//         N = 3  EC, HLLD, PP       1458 55.3 -> 49.6   2000 56.1 -> 57.8
//         N = 4  EC, Rusanov, PP    1463 56.4 -> 47.7   2048 58.7 -> 59.1
// HLLD at N = 4 takes this form at any size (10976 blocks: FP64 1133 -> 833,
// FP32 825 -> 364): there stage_kernel keeps the terms of three directions'
// code in one register allocation and spills 1 to 2 KB per lane.
template <int M, typename Real>
long long wide_blocks(const nemo_gpu_config& c) {
    constexpr bool F32 = sizeof(Real) == 4;
    const bool ec = c.volume == NEMO_VOL_EC;
    if (c.equations == NEMO_EQ_GLM_MHD) {
        if (M == 5 && c.surface == NEMO_SURF_HLLD) return INT64_MAX;
        if (!F32) return 400;
        return M == 3 ? (ec ? 1200 : 1024) : 1536;
    }
    return EULER_WIDE[F32][M - 3][ec][c.surface == NEMO_SURF_HLLC][c.indicator == NEMO_IND_PP]
                     [c.timedisc == NEMO_TD_SSPRK54];
}

// Whether a launch over nblocks blocks takes the small-mesh form; `form` is
// NEMO_FORM_AUTO or one of the two.
template <int M, typename Real>
bool wide_form(const nemo_gpu_config& c, int form, long long nblocks) {
    return form == NEMO_FORM_AUTO ? nblocks <= wide_blocks<M, Real>(c) : form == NEMO_FORM_FOUR_WAVES;
}

}  // namespace nemo_host
