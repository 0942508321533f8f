// The NUFFT runs' part of the reverse sweep (nufft_back.hip), launched by hb_adjoint_runs (adjoint.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/blochparty_amd.h"

namespace hb {

// Runs [r0, r1) of an interval. m0: (r1 - r0, 2, n_pad) Mx, My at each run's start; q: (r1 - r0, 2, n_pad) what the
// run's samples add to lambda there; g: (5 + 2 nc, n_pad) float64 accumulators of dL/d(R2, px, py, pz, db0) and, with
// coil_grads, of the coil gradients, each run added in turn, last first.
struct NufftBack {
    const float* m0;
    float* q;
    double* g;
    int n_pad, r0, r1, coil_grads;
};

// Whether the kernel takes nc coils and windows of up to cols columns.
bool nufft_back_takes(int nc, int cols);
void launch_nufft_back(const NufftBack& a, const hb_case& cs, const hb_adjoint& ad, const int32_t* heads,
                       hipStream_t st);

}  // namespace hb
