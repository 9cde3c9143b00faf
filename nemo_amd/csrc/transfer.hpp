// State transfers between the host arrays u[elem][var][node] (the reference's
// per-quad layout) and the device layout u[var][elem][node], shared by the
// single-mesh solver and the batched ensemble.
#pragma once

#include <hip/hip_runtime.h>

namespace nemo_host {

// Elements [off, off + ne) of a device state of `stride` elements per
// variable to the host array `host`.  `scratch` holds V*ne*M3 doubles on the
// device; its content is lost.  Returns when the host array is complete.
hipError_t state_to_host(hipStream_t stream, const double* dev, long long stride, long long off, long long ne, int V,
                         int M3, double* scratch, double* host);

// The reverse.  The host array may be reused on return; the device state is
// complete in stream order.
hipError_t state_to_device(hipStream_t stream, const double* host, double* scratch, double* dev, long long stride,
                           long long off, long long ne, int V, int M3);

// Every handle holds the staging buffers' process-wide share while it lives;
// they are freed with the last one.
void staging_retain();
void staging_release();

// 64 bytes of pinned host memory that kernels write their reports to; nullptr
// if there is none to be had.
void* report_get();
void report_put(void* p);

}  // namespace nemo_host
