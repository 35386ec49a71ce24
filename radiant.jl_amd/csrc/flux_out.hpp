// flux_out.hpp -- flux moments [G][Np][Nc] on the device into host memory in Radiant's layout
// [Nc][Np][G] (group fastest), on stream st; returns once the caller's memory is complete.
#pragma once
#include <hip/hip_runtime.h>

namespace rt {
void flux_to_host(double* out, const double* phi, int G, int Np, int Nc, hipStream_t st);
}
