// Adjoint (gradient of sum_b w_b P0_b w.r.t. positions) and grid interpolation at positions.
#pragma once
#include "common.hpp"

namespace pyl {

// grad[3p + a] = scale * (N/L) * sum_cells G * W'_a prod W_b  (float32 grid G, (n,3) output)
int gather_grad(const float* G, int N, double BoxSize, const float* pos, int64_t n, int scheme, double scale,
                float* grad, hipStream_t st);

// out[p] = sum_cells G * prod W  (MAS_library.CIC_interp with scheme 2)
int interp(const float* G, int N, double BoxSize, const float* pos, int64_t n, int scheme, float* out,
           hipStream_t st);

}  // namespace pyl
