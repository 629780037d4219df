// Conservative ray/surfel test shared by the render and its backward.
#pragma once

#include <hip/hip_runtime.h>

namespace nest {

// Conservative form of the exact ray/surfel tests (splat_hit, bwd_hit), for the
// passes that list a pixel's candidates: an rcp-based rho3d within 1e-6 of the exact one, scaled down by
// 1e-5, above the splat's cut and rho2d above it too means alpha < 1/255 in
// the exact test.  False only for such pairs; NaNs are candidates.
__device__ __forceinline__ bool splat_near(float4 q0, float4 q1, float4 q2, float cut, float pxf, float pyf) {
  const float Tu0 = q0.x, Tu1 = q0.y, Tu2 = q0.z, Tv0 = q0.w;
  const float Tv1 = q1.x, Tv2 = q1.y, Tw0 = q1.z, Tw1 = q1.w;
  const float Tw2 = q2.x;
  const float k0 = pxf * Tw0 - Tu0, k1 = pxf * Tw1 - Tu1, k2 = pxf * Tw2 - Tu2;
  const float l0 = pyf * Tw0 - Tv0, l1 = pyf * Tw1 - Tv1, l2 = pyf * Tw2 - Tv2;
  const float p0 = k1 * l2 - k2 * l1, p1 = k2 * l0 - k0 * l2, p2 = k0 * l1 - k1 * l0;
  const float dx = q2.y - pxf, dy = q2.z - pyf;
  const float rho2d = 2.0f * (dx * dx + dy * dy);
  const float rc = __builtin_amdgcn_rcpf(p2);
  const float sxa = p0 * rc, sya = p1 * rc;
  return !((sxa * sxa + sya * sya) * 0.99999f > cut && rho2d > cut);
}

}  // namespace nest
