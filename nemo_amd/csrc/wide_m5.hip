// Small-mesh stage kernels of n_poly = 4 (M = 5 nodes per direction), gfx950.
#include "stage_wide_launch.hpp"

namespace nemo_host {
template int launch_wide<5, double>(Solver& s, const nemo::StageArgs<5, double>& a, bool net);
template int launch_wide<5, float>(Solver& s, const nemo::StageArgs<5, float>& a, bool net);
}  // namespace nemo_host
