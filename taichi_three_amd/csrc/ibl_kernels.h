// ibl_kernels.h -- prefiltered environment maps for image-based lighting.
//
//   k_bake_ibl  Lambert.cook_for_ibl (tina/matr/material.py:407-438) and
//               CookTorrance.cook_for_ibl (material.py:279-320): each
//               output texel's direction from Skybox.unmapcoor
//               (tina/skybox.py:131-136), nsamples directions around it in
//               tangentspace (tina/advans.py:96-108), each weighted by its
//               cosine u; out = sum(env(dir) * u) / sum(u).
//
// The reference draws (u, v) from ti.random and denoises the Lambert map with a
// KNN filter.  Here the points are the Hammersley set ((s + 0.5)/n, radical
// inverse of s), so a bake is a deterministic function of the environment and
// needs no denoiser, and the arithmetic is binary64 with the sample sum taken
// in a fixed order.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "shade_dev.h"

namespace tina {

struct D3 { double x, y, z; };
__device__ __forceinline__ D3 d3(double x, double y, double z) { return D3{x, y, z}; }
__device__ __forceinline__ D3 dsmul(double s, D3 a) { return d3(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ double ddot(D3 a, D3 b) { return ((a.x * b.x) + (a.y * b.y)) + (a.z * b.z); }
__device__ __forceinline__ D3 dcross(D3 a, D3 b) {
  return d3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
// Matrix.normalized(): v * (1 / sqrt(v.v))
__device__ __forceinline__ D3 dnormalized(D3 a) { return dsmul(1.0 / sqrt(ddot(a, a)), a); }

// Skybox.sample (tina/skybox.py:23-28, 138-145; bilerp, tina/common.py:140-149)
// of a [w][h][3] f32 equirect map, indices clamped to the map, as its four
// texels and their weights, the weights times k.  sky_fetch issues the loads and
// sky_add consumes them, so that several samples' loads are in flight at once.
struct SkyTap {
  double w[4];
  V3 t[4];
};

__device__ __forceinline__ void sky_fetch(gf32* __restrict__ img, int w, int h, D3 dir, double k, SkyTap& s) {
  const double p = atan2(-dir.z, dir.x) * 0.15915494309189535;  // 1 / tau
  const double px = (double)(w - 1) * (p - floor(p));
  const double py = (double)(h - 1) * __builtin_fma(dir.y, 0.5, 0.5);
  // clamped before the conversion: a NaN becomes texel 0 (its weights stay NaN)
  const double fx = fmin(fmax(floor(px), 0.0), (double)(w - 1)), fy = fmin(fmax(floor(py), 0.0), (double)(h - 1));
  const int xa = (int)fx, ya = (int)fy;
  const int xb = min(xa + 1, w - 1), yb = min(ya + 1, h - 1);
  gf32* ca = img + (size_t)xa * h * 3;
  gf32* cb = img + (size_t)xb * h * 3;
  s.t[0] = ld3(ca + 3 * ya);
  s.t[1] = ld3(ca + 3 * yb);
  s.t[2] = ld3(cb + 3 * ya);
  s.t[3] = ld3(cb + 3 * yb);
  const double x0 = px - fx, x1 = py - fy;
  const double k1 = k * x0, k0 = k - k1;
  s.w[3] = k1 * x1;
  s.w[2] = k1 - s.w[3];
  s.w[1] = k0 * x1;
  s.w[0] = k0 - s.w[1];
}

__device__ __forceinline__ void sky_add(const SkyTap& s, D3& r) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    r.x = __builtin_fma(s.w[i], (double)s.t[i].x, r.x);
    r.y = __builtin_fma(s.w[i], (double)s.t[i].y, r.y);
    r.z = __builtin_fma(s.w[i], (double)s.t[i].z, r.z);
  }
}

// Van der Corput radical inverse in base 2 (bit reversal of s, scaled by 2^-32)
__device__ __forceinline__ double radical_inverse2(uint32_t s) {
  return (double)__builtin_bitreverse32(s) * 2.3283064365386963e-10;
}

// Skybox.unmapcoor + unspheremap + spherical (tina/skybox.py:31-35, 131-136;
// tina/advans.py:104-108) for texel (ix, iy) of a w x h map
__device__ __forceinline__ D3 unmapcoor_f64(int ix, int iy, int w, int h) {
  const double tau = 6.283185307179586;
  const double v = (double)ix / (double)(w - 1), u = (double)iy / (double)(h - 1);
  const double hh = u * 2.0 - 1.0;
  const double r = sqrt(fmax(0.0, 1.0 - hh * hh));
  const double dx = r * cos(v * tau), dy = r * sin(v * tau), dz = hh;
  return d3(dx, dz, -dy);
}

// A bake workgroup: kBakeBlock lanes as `tpb` texels (a power of two, at most
// 64) by kBakeBlock / tpb sample slices.
//
// What bounds a bake is binary64 arithmetic (162 VALU instructions a sample, 110
// of them in atan2).  The samples' own part -- the cosine u, its sine and the
// cos / sin of the azimuth, which depend on the sample alone -- is worked out
// once per workgroup, a lane a sample, into LDS and read back by every texel.
// The slices give the coarse levels (a 512 x 256 sky's irradiance map is 3,528
// texels of 4,096 samples) enough lanes to fill the chip, and are summed by a
// fixed tree.  The seven maps of that sky at precision 32 (101 M samples):
// 11.86 ms with a lane a texel and everything per sample, 0.67 ms so; one
// sample at a time instead of two in flight (its four loads were then waited for
// one by one): 1.14 ms.
constexpr int kBakeBlock = 512;

// Texels a workgroup.  A wave whose lanes all take one sample reads neighbouring
// texels, so as many as 64 while that leaves two workgroups a CU (what it
// holds) and 16 at least; fewer only to get a workgroup for most CUs.  Measured
// at 64 / 32 / 16 / 8 / 4 / 2 texels: 110,450 texels x 256 samples 168 / 189 / 219
// / 279 / 393 / 656 us; 18,818 x 560 113 / 88 / 82 / 90 / 115 / 181; 3,528 x 4,096
// 378 / 212 / 153 / 172 / 168 / 169; 450 x 4,423 391 / 206 / 115 / 70 / 47 / 37.
inline int bake_tpb(long texels, int ncu) {
  int tpb = 64;
  while (tpb > 1 && (texels + tpb - 1) / tpb < (tpb > 16 ? 2L * ncu : 4L * ncu / 5)) tpb >>= 1;
  return tpb;
}

// alpha2 < 0 selects the cosine (Lambert) bake; otherwise the GGX-distributed
// cosines u = sqrt((1 - u0) / (1 - u0 (1 - alpha2))) of CookTorrance.cook_for_ibl.
__global__ void __launch_bounds__(kBakeBlock) __attribute__((amdgpu_waves_per_eu(4))) k_bake_ibl(const float* __restrict__ env, int ew, int eh,
                                                         float* __restrict__ out, int ow, int oh, double alpha2,
                                                         int nsamples, int tpb) {
  // a chunk's samples: u, r cos, r sin (tina/advans.py:104-108); then the slices' sums
  __shared__ double s_u[kBakeBlock], s_x[kBakeBlock], s_y[kBakeBlock], s_d[kBakeBlock];
  const int tid = threadIdx.x, slices = kBakeBlock / tpb, slice = tid / tpb;
  const long t = (long)blockIdx.x * tpb + tid % tpb, n_tex = (long)ow * oh;
  gf32* e = gptr((uint64_t)env);
  const long tc = t < n_tex ? t : n_tex - 1;
  const D3 nrm = unmapcoor_f64((int)(tc / oh), (int)(tc % oh), ow, oh);
  // tangentspace(nrm) (tina/advans.py:96-100)
  const D3 bitan = dnormalized(dcross(nrm, d3(233.0, 666.0, 512.0)));
  const D3 tan = dcross(bitan, nrm);
  D3 res = d3(0.0, 0.0, 0.0);
  double dem = 0.0;
  const double n = (double)nsamples, tau = 6.283185307179586;
  for (long c0 = 0; c0 < nsamples; c0 += kBakeBlock) {
    const int m = (int)min((long)kBakeBlock, nsamples - c0);
    __syncthreads();  // the previous chunk is consumed
    if (tid < m) {
      const uint32_t s = (uint32_t)(c0 + tid);
      const double u0 = ((double)s + 0.5) / n, a = radical_inverse2(s) * tau;
      const double u = alpha2 < 0.0 ? u0 : sqrt((1.0 - u0) / (1.0 - u0 * (1.0 - alpha2)));
      const double r = sqrt(fmax(0.0, 1.0 - u * u));
      s_u[tid] = u;
      s_x[tid] = r * cos(a);
      s_y[tid] = r * sin(a);
    }
    __syncthreads();
    auto fetch = [&](int i, SkyTap& q) {
      const double u = s_u[i], sx = s_x[i], sy = s_y[i];
      const D3 d = d3(__builtin_fma(u, nrm.x, __builtin_fma(sy, bitan.x, sx * tan.x)),
                      __builtin_fma(u, nrm.y, __builtin_fma(sy, bitan.y, sx * tan.y)),
                      __builtin_fma(u, nrm.z, __builtin_fma(sy, bitan.z, sx * tan.z)));
      sky_fetch(e, ew, eh, d, u, q);
    };
    // two samples at a time: both samples' loads go out before the first is used
    for (int i = slice; i < m; i += 2 * slices) {
      const bool two = i + slices < m;
      SkyTap q0, q1;
      fetch(i, q0);
      fetch(two ? i + slices : i, q1);
      __builtin_amdgcn_sched_barrier(0);
      sky_add(q0, res);
      dem += s_u[i];
      if (two) {
        sky_add(q1, res);
        dem += s_u[i + slices];
      }
    }
  }
  __syncthreads();
  s_u[tid] = res.x;
  s_x[tid] = res.y;
  s_y[tid] = res.z;
  s_d[tid] = dem;
  for (int half = slices / 2; half > 0; half >>= 1) {
    __syncthreads();
    if (slice < half) {
      const int o = tid + half * tpb;
      s_u[tid] += s_u[o];
      s_x[tid] += s_x[o];
      s_y[tid] += s_y[o];
      s_d[tid] += s_d[o];
    }
  }
  // slice 0's own sums: written by this lane
  if (slice == 0 && t < n_tex) {
    float* o = out + t * 3;
    o[0] = (float)(s_u[tid] / s_d[tid]);
    o[1] = (float)(s_x[tid] / s_d[tid]);
    o[2] = (float)(s_y[tid] / s_d[tid]);
  }
}

}  // namespace tina
