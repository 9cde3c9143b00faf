// Stage kernels of n_poly = 4 (M = 5 nodes per direction), gfx950.
#include "stage_launch.hpp"

namespace nemo_host {
template bool takes_wide<5>(const Solver& s, const LaunchOpts& o);
template int launch_stage_m<5>(Solver& s, int stage, double dt, const double* dt_dev, double* rhs_out,
                                double* alpha_out, double* cfl_part, const LaunchOpts& o);
}  // namespace nemo_host
