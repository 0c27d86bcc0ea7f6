// The Hessian factor record of the factored route (k_hfactors in plain.hip):
// per element [M_q (9 per point) | cl_q | cc_q | w mu jit jit^T (6)], padded
// to a multiple of 4 values.
#pragma once

namespace pfgpu {

__host__ __device__ constexpr int fac_size(int nq) { return (11 * nq + 6 + 3) & ~3; }

} // namespace pfgpu
