// Shared pieces of the v1 sampler (phitest/render/cuda/src/sampling.hpp):
// mip level pointers, level selection, and the sample position and LoD of
// samplePos3D for the four coordinate modes. Used by the resample ops and the
// batched mipmapped render.
#pragma once
#include "gft_device.hpp"

namespace gft {

__device__ __forceinline__ const float* level_ptr(const float* base, const float* atlas, const MipTable& mt, int b,
                                                  int m) {
  return m == 0 ? base + (size_t)b * mt.base_stride : atlas + (size_t)b * mt.atlas_stride + mt.offset[m];
}
__device__ __forceinline__ float* level_ptr_mut(float* base, float* atlas, const MipTable& mt, int b, int m) {
  return m == 0 ? base + (size_t)b * mt.base_stride : atlas + (size_t)b * mt.atlas_stride + mt.offset[m];
}

// Mip level selection (sampling.hpp:551-571,603-620): returns the number of
// taps (1 or 2) with their levels and weights.
__device__ __forceinline__ int level_taps(const SampleCfg& s, float lod, int* lv, float* w) {
  if (s.mm == MIP_NONE) {
    lv[0] = 0;
    w[0] = 1.f;
    return 1;
  }
  float l = fminf(fmaxf(lod + s.bias, 0.f), (float)s.levels);
  int fl = min((int)(l + (s.mm == MIP_NEAREST ? 0.5f : 0.f)), s.levels);
  if (s.mm == MIP_LINEAR) {
    int cl = min((int)ceilf(l), s.levels);
    if (cl > fl) {
      float fr = l - floorf(l);
      lv[0] = fl;
      w[0] = 1.f - fr;
      lv[1] = cl;
      w[1] = fr;
      return 2;
    }
  }
  lv[0] = fl;
  w[0] = 1.f;
  return 1;
}

// 2^-m
__device__ __forceinline__ float level_scale(int m) { return __int_as_float((127 - m) << 23); }

// 1 / w to within an ulp: the hardware's estimate and one Newton step
__device__ __forceinline__ float recip(float w) {
  const float r = __builtin_amdgcn_rcpf(w);
  return fmaf(fmaf(-w, r, 1.f), r, r);
}

// n / w with r = recip(w): the product, corrected twice by its residual
// (Markstein's method for a fused multiply-add), without a float division's
// scaling, which only quotients and divisors beyond 2^+-96 need; zeros, infinities
// and NaN come out as in a division. Several numerators share a reciprocal.
__device__ __forceinline__ float quotient(float n, float w, float r) {
  float q = n * r;
  q = fmaf(fmaf(-w, q, n), r, q);
  q = fmaf(fmaf(-w, q, n), r, q);
  return __builtin_amdgcn_div_fixupf(q, w, n);
}

// Input position of output index q (+ 0.5) in the reverse modes
// (sampling.hpp:59-136); w is the projected W, vz the view depth.
__device__ __forceinline__ float3 map_reverse(const ReverseMap& v, int cm, float qx, float qy, float qz, float& w,
                                              float& vz) {
  const float4 vs = mat_vec(v.A, qx, qy, qz, 1.f);
  const float4 ndc = mat_vec(v.B, vs.x, vs.y, vs.z, vs.w);
  const float rw = recip(ndc.w);
  const float ndx = quotient(ndc.x, ndc.w, rw), ndy = quotient(ndc.y, ndc.w, rw), ndz = quotient(ndc.z, ndc.w, rw);
  float3 r = make_float3((ndx * 0.5f + 0.5f) * v.idims[0], (ndy * 0.5f + 0.5f) * v.idims[1],
                         (ndz * 0.5f + 0.5f) * v.idims[2]);
  w = ndc.w;
  vz = 0.f;
  if (cm == CM_LINDEPTH_REVERSE) {
    const float range = v.farp - v.nearp;
    vz = quotient(-v.p32, ndz + v.p22, recip(ndz + v.p22));
    const float t = quotient(-(vz + v.nearp), range, recip(range));
    r.z = t * v.idims[2];
  }
  return r;
}

__device__ __forceinline__ float len3f(float a, float b, float c) { return sqrtf(a * a + b * b + c * c); }

// Input position (and with LOD its level of detail) of output index q (+ 0.5):
// the coordinate maps of samplePos3D (sampling.hpp:59-136). The level of detail
// is log2 of the largest footprint of the forward differences p(q) - p(q +
// e_j): Jacobian rows for the forward modes, columns for the reverse modes. In
// the forward modes the differences are formed directly, p(q) - p(q + e) = (p gW
// - g) / (W + gW) with g the forms' change, not from four positions.
template <bool LOD>
__device__ __forceinline__ float3 map_sample(const SampleView& v, int cm, float qx, float qy, float qz, float& lod) {
  const bool lin = cm == CM_LINDEPTH;
  lod = 0.f;
  if (!lin && cm != CM_TRANSFORM) {
    float w, vz;
    const float3 p = map_reverse(v.rev, cm, qx, qy, qz, w, vz);
    if constexpr (LOD) {
      const float3 a = map_reverse(v.rev, cm, qx + 1.f, qy, qz, w, vz);
      const float3 b = map_reverse(v.rev, cm, qx, qy + 1.f, qz, w, vz);
      const float3 c = map_reverse(v.rev, cm, qx, qy, qz + 1.f, w, vz);
      const float fx = len3f(p.x - a.x, p.y - a.y, p.z - a.z), fy = len3f(p.x - b.x, p.y - b.y, p.z - b.z),
                  fz = len3f(p.x - c.x, p.y - c.y, p.z - c.z);
      lod = fmaxf(0.f, log2f(fmaxf(fx, fmaxf(fy, fz))));
    }
    return p;
  }
  const float x = qx - v.mid[0], y = qy - v.mid[1], z = qz - v.mid[2];
  const float s = lin ? fmaf(v.z1, z, v.z0) : 1.f;
  float E[4], h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i == 3 && v.unit) {
      E[i] = 0.f;
      h[i] = 1.f;
      break;
    }
    E[i] = fmaf(v.b[i], y, fmaf(v.a[i], x, v.e[i]));
    h[i] = lin ? fmaf(E[i], s, v.c[i]) : fmaf(v.c[i], z, E[i]);
  }
  float3 p = make_float3(h[0], h[1], h[2]);
  if (!v.unit) {
    const float r = recip(h[3]);
    p.x *= r;
    p.y *= r;
    p.z *= r;
  }
  if constexpr (LOD) {
    float f[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      // the forms' change along output axis j
      float g[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float k = j == 0 ? v.a[i] : (j == 1 ? v.b[i] : v.c[i]);
        g[i] = lin ? (j == 2 ? E[i] * v.z1 : k * s) : k;
      }
      float d[3] = {-g[0], -g[1], -g[2]};
      if (!v.unit) {
        const float r = recip(h[3] + g[3]);
        d[0] = fmaf(p.x, g[3], d[0]) * r;
        d[1] = fmaf(p.y, g[3], d[1]) * r;
        d[2] = fmaf(p.z, g[3], d[2]) * r;
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) f[i] = fmaf(d[i], d[i], f[i]);
    }
    // log2 of the norm; a subnormal square is below level 0 anyway
    lod = fmaxf(0.f, 0.5f * __builtin_amdgcn_logf(fmaxf(f[0], fmaxf(f[1], f[2]))));
  }
  return p;
}

__device__ __forceinline__ float3 map_pos(const SampleView& v, int cm, float qx, float qy, float qz) {
  float l;
  return map_sample<false>(v, cm, qx, qy, qz, l);
}

}  // namespace gft
