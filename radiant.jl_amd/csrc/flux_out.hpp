// flux_out.hpp -- flux moments [G][Np][Nc] on the device into host memory in Radiant's layout
// [Nc][Np][G] (group fastest), on stream st; returns once the caller's memory is complete.
#pragma once
#include <hip/hip_runtime.h>

namespace rt {
// Into the pinned ring by the rearranging kernels, by the copy engines (for a device that other work
// keeps busy), or without the ring.  The same values each way.
enum FluxWay { FLUX_LINK = 0, FLUX_ENGINE = 1, FLUX_DIRECT = 2 };
// Device memory that the copy engines' way may write: two blocks of n doubles (below 1 MiB it goes without)
struct FluxScratch { double* p[2]; size_t n; };
void flux_to_host(double* out, const double* phi, int G, int Np, int Nc, FluxWay way, const FluxScratch& scratch,
                  hipStream_t st);
// Copies a host array through the device and out again (test hook behind rt_test_flux_out).
void test_flux_out(int way, int G, int Np, int Nc, const double* phi, size_t chunk, double* out);
}
