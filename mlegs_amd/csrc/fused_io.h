// Fields of the fused products kernels (k_fused.hip, k_fused_any.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace mlg {
struct FusedIO {
  const double2 *in[10];  // rur rup uz ror rop oz rbr rbp bz [W]
  double2 *out[4];        // r N_r, r N_theta, N_z, N_b (PFP)
  double *zl;             // an LN coefficient the launch sets to zero (N_b's), or null
};
}  // namespace mlg
