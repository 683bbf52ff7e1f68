// Host-side helpers of the C ABI: thread-local error reporting, shape
// validation in the reference's wording, and camera-record packing.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <string>
#include <vector>

#include "gft_device.hpp"
#include "../../include/gft.h"

namespace gft {

void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);
int check_hip(hipError_t e, const char* what);

// Column-major 4x4 in double; m[4*col + row]
struct Mat4d {
  double m[16];
};
Mat4d mat_from_colmajor(const float* a);
Mat4d mat_identity();
Mat4d mat_mul(const Mat4d& a, const Mat4d& b);
bool mat_inverse(const Mat4d& a, Mat4d& out);
void mat_to_float(const Mat4d& a, float* out);

// The (batch, camera) pairs an op visits, in the reference's launch order
// (batch-major; all cameras per batch when separate_camera_batch, camera b for
// batch b otherwise).
struct ViewPair {
  int batch, cam, slot;
};
std::vector<ViewPair> view_pairs(int N, int num_cameras, bool separate_camera_batch);

// Pixels that look through a unit of the x-, y- and z-facing area of grid d at
// its centre, in an image of w x h pixels: the cross products of the pixel
// coordinates' derivatives along the grid's axes. A is projection * model-view,
// column-major. False where the centre has no finite image.
template <class T> bool face_pixels(const T* A, Dims3 d, double w, double h, double n[3]) {
  const double x = 0.5 * d.x, y = 0.5 * d.y, z = 0.5 * d.z;
  auto row = [&](int r) { return A[r] * x + A[4 + r] * y + A[8 + r] * z + A[12 + r]; };
  const double cx = row(0), cy = row(1), cw = row(3);
  double gx[3], gy[3];
  for (int a = 0; a < 3; ++a) {
    gx[a] = 0.5 * w * (A[4 * a] * cw - cx * A[4 * a + 3]) / (cw * cw);
    gy[a] = 0.5 * h * (A[4 * a + 1] * cw - cy * A[4 * a + 3]) / (cw * cw);
  }
  for (int a = 0; a < 3; ++a) {
    const int b = (a + 1) % 3, c = (a + 2) % 3;
    n[a] = std::fabs(gx[b] * gy[c] - gx[c] * gy[b]);
  }
  return std::isfinite(n[0] + n[1] + n[2]);
}

// Per-view projective coefficients of the raymarch's pixel rays (near0, far0,
// gx, gy of ProjView) from the inverse projection and inverse model-view.
void ray_coefficients(const Mat4d& pinv, const Mat4d& mvinv, const RayDims& rd, ProjView& pv);

}  // namespace gft
