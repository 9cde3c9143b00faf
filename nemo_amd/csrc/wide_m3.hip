// Small-mesh stage kernels of n_poly = 2 (M = 3 nodes per direction), gfx950.
#include "stage_wide_launch.hpp"

namespace nemo_host {
template int launch_wide<3, double>(Solver& s, const nemo::StageArgs<3, double>& a, bool net);
template int launch_wide<3, float>(Solver& s, const nemo::StageArgs<3, float>& a, bool net);
}  // namespace nemo_host
