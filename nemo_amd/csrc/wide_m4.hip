// Small-mesh stage kernels of n_poly = 3 (M = 4 nodes per direction), gfx950.
#include "stage_wide_launch.hpp"

namespace nemo_host {
template int launch_wide<4, double>(Solver& s, const nemo::StageArgs<4, double>& a, bool net);
template int launch_wide<4, float>(Solver& s, const nemo::StageArgs<4, float>& a, bool net);
}  // namespace nemo_host
