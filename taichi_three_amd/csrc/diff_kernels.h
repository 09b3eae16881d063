// diff_kernels.h -- differentiable deferred shading and its adjoint.
//
// The material is Tina's PBR (tina/matr/material.py:322-362, 387-396, 701-706)
// under point lights (tina/core/lighting.py:84-98), with albedo, smooth normal,
// roughness and metallic interpolated per vertex of an indexed mesh and a scalar
// intensity per light.  Visibility comes from the packed depth|id buffer of
// the raster pass and is held fixed (no gradient through coverage).
//
//   k_dshade_fwd  colour of every covered pixel
//   k_dshade_bwd  given dLoss/dcolour per pixel: recomputes the face's
//                 perspective-correct weights from the saved id buffer (nothing
//                 per pixel is stored by the forward pass), walks the shading
//                 backwards by hand (diff_adjoint), applies the normalisation and
//                 interpolation Jacobians and adds the result to the three
//                 vertices, first in LDS per block of pixels, then with float
//                 atomics; light-intensity gradients are summed per workgroup.
#pragma once
#include "shade_kernels.h"

namespace tina {

// ---- the shaded colour ------------------------------------------------------------

struct DiffArgs {
  Cam cam;
  uint64_t soup;     // [F][3][3] f32 positions (the raster's input)
  uint64_t faces;    // [F][3] i32 vertex indices
  uint64_t nrm, col; // [V][3] f32
  uint64_t rough, metal;  // [V] f32
  uint64_t inten;    // [L] f32
  int nfaces;
  uint32_t id_base;
  int nlights;
  float lpos[TINA_MAX_LIGHTS][3];
  float lcol[TINA_MAX_LIGHTS][3];
  float amb[3];
  float f0_dielectric;  // 0.16 specular^2
};

// PBR under the point lights for one pixel: albedo a, unit normal n, roughness r,
// metallic m, at position pos seen from V.
__device__ __forceinline__ V3 diff_color(const DiffArgs& A, gf32* inten, V3 a, V3 n, float r, float m, V3 pos, V3 V) {
  const float inv_pi = (float)(1.0 / 3.141592653589793);
  const float EPS = 1e-10f, ONE_M_EPS = (float)(1.0 - 1e-10);
  // f0 = m a + (1 - m) 0.16 spec^2 ; PBR = Mix(Lambert a, CT(r, f0), f0)
  const float om = 1.0f - m;
  const V3 f0 = v3(m * a.x + om * A.f0_dielectric, m * a.y + om * A.f0_dielectric, m * a.z + om * A.f0_dielectric);
  // ambient: amb * ((1 - f0) a + f0)
  V3 c = v3(A.amb[0] * ((1.0f - f0.x) * a.x + f0.x), A.amb[1] * ((1.0f - f0.y) * a.y + f0.y),
            A.amb[2] * ((1.0f - f0.z) * a.z + f0.z));
  const float r2 = fmaxf(1e-6f, r * r);
  const float k = 0.5f * r2;
  for (int l = 0; l < A.nlights; l++) {
    V3 L = v3(A.lpos[l][0] - pos.x, A.lpos[l][1] - pos.y, A.lpos[l][2] - pos.z);
    const float dist = sqrtf(vdot(L, L));
    L = vdivs(L, dist);
    const float cosv = vdot(n, L);
    if (!(cosv > 0.0f)) continue;
    const V3 h = vnormalized(vadd(L, V));
    const float NoH = fmaxf(EPS, vdot(n, h));
    const float NoL = fmaxf(EPS, cosv);
    const float NoV = fmaxf(EPS, vdot(n, V));
    const float VoH = fminf(ONE_M_EPS, fmaxf(EPS, vdot(h, V)));
    const float den = 1.0f - (NoH * NoH) * (1.0f - r2);
    const float ndf = fdiv_rn(r2, den * den);
    const float vdf = fdiv_rn(fdiv_rn(1.0f, (NoV * k + 1.0f) - k) * fdiv_rn(1.0f, (NoL * k + 1.0f) - k),
                              (1.0f - r2) + (float)(4.0 * 3.141592653589793) * r2);
    const float x1 = 1.0f - VoH, x2 = x1 * x1, p5 = (x2 * x2) * x1;
    const float nv = ndf * vdf;
    const float sc = fdiv_rn(1.0f, dist * dist);
    const V3 br = v3((1.0f - f0.x) * a.x * inv_pi + f0.x * nv * (f0.x + p5 * (1.0f - f0.x)),
                     (1.0f - f0.y) * a.y * inv_pi + f0.y * nv * (f0.y + p5 * (1.0f - f0.y)),
                     (1.0f - f0.z) * a.z * inv_pi + f0.z * nv * (f0.z + p5 * (1.0f - f0.z)));
    const float I = inten[l];
    c.x = c.x + I * (cosv * ((A.lcol[l][0] * sc) * br.x));
    c.y = c.y + I * (cosv * ((A.lcol[l][1] * sc) * br.y));
    c.z = c.z + I * (cosv * ((A.lcol[l][2] * sc) * br.z));
  }
  return c;
}

// The gradients of one pixel.
struct DiffGrad {
  V3 a, n;     // albedo, unit normal
  float r, m;  // roughness, metallic
};

// dLoss/d(albedo, normal, roughness, metallic) from g = dLoss/dcolour: diff_color
// walked backwards, light by light, with its intermediates recomputed.  Light
// l's g . du / dintensity goes to light(l, value), also for a pixel with no face
// (live false: every gradient 0), so that a wave may reduce it.
template <class PerLight>
__device__ __forceinline__ DiffGrad diff_adjoint(const DiffArgs& A, gf32* inten, V3 a, V3 n, float r, float m, V3 pos,
                                                 V3 V, V3 g, bool live, PerLight&& light) {
  const float inv_pi = (float)(1.0 / 3.141592653589793);
  const float EPS = 1e-10f, ONE_M_EPS = (float)(1.0 - 1e-10), c3 = (float)(4.0 * 3.141592653589793);
  const float om = 1.0f - m, d0 = A.f0_dielectric;
  const V3 f0 = v3(m * a.x + om * d0, m * a.y + om * d0, m * a.z + om * d0);
  const V3 of = vsub(vs(1.0f), f0), amb = v3(A.amb[0], A.amb[1], A.amb[2]);
  const bool r_free = r * r > 1e-6f;  // max(1e-6, r^2) takes r^2
  const float r2 = fmaxf(1e-6f, r * r), k = 0.5f * r2, om2 = 1.0f - r2;
  const float nov = vdot(n, V), NoV = fmaxf(EPS, nov);
  const float ia1 = fdiv_rn(1.0f, (NoV * k + 1.0f) - k), ia3 = fdiv_rn(1.0f, om2 + c3 * r2);
  const V3 ga_amb = vmul(g, amb);
  DiffGrad q;
  q.a = vmul(ga_amb, of);                       // ambient: (1 - f0) a + f0
  V3 gf0 = vmul(ga_amb, vsub(vs(1.0f), a));
  q.n = vs(0.0f);
  float gr2 = 0.0f, gnov = 0.0f;
  for (int l = 0; l < A.nlights; l++) {
    V3 L = v3(A.lpos[l][0] - pos.x, A.lpos[l][1] - pos.y, A.lpos[l][2] - pos.z);
    const float dist = sqrtf(vdot(L, L));
    L = vdivs(L, dist);
    const float cosv = vdot(n, L);
    float gi = 0.0f;
    if (live && cosv > 0.0f) {
      const V3 h = vnormalized(vadd(L, V));
      const float noh = vdot(n, h), NoH = fmaxf(EPS, noh), NoL = fmaxf(EPS, cosv);
      const float VoH = fminf(ONE_M_EPS, fmaxf(EPS, vdot(h, V)));
      const float iden = fdiv_rn(1.0f, 1.0f - (NoH * NoH) * om2), iden2 = iden * iden;
      const float ndf = r2 * iden2;
      const float ia2 = fdiv_rn(1.0f, (NoL * k + 1.0f) - k);
      const float vdf = (ia1 * ia2) * ia3;
      const float x1 = 1.0f - VoH, x2 = x1 * x1, p5 = (x2 * x2) * x1;
      const float nv = ndf * vdf, sc = fdiv_rn(1.0f, dist * dist), I = inten[l];
      const V3 F = vadd(f0, vsmul(p5, of));     // Fresnel
      const V3 br = vadd(vsmul(inv_pi, vmul(of, a)), vsmul(nv, vmul(f0, F)));
      // u = cosv K br, K = light colour / dist^2; c += I u
      const V3 gk = v3(g.x * (A.lcol[l][0] * sc), g.y * (A.lcol[l][1] * sc), g.z * (A.lcol[l][2] * sc));
      const float gkb = vdot(gk, br);
      gi = gkb * cosv;
      float gcos = I * gkb;
      const V3 gbr = vsmul(I * cosv, gk);
      q.a = vadd(q.a, vsmul(inv_pi, vmul(gbr, of)));
      // d br / d f0 = nv (F + f0 (1 - p5)) - a / pi
      gf0 = vadd(gf0, vmul(gbr, vsub(vsmul(nv, vadd(F, vsmul(1.0f - p5, f0))), vsmul(inv_pi, a))));
      const float gnv = vdot(gbr, vmul(f0, F));
      // ndf = r2 / den^2, den = 1 - NoH^2 (1 - r2)
      const float gndf = gnv * vdf, t = ((2.0f * ndf) * iden) * gndf;  // -dLoss/dden
      gr2 = gr2 + (gndf * iden2 - t * (NoH * NoH));
      if (noh > EPS) q.n = vadd(q.n, vsmul((2.0f * t) * (NoH * om2), h));
      // vdf = 1 / (a1 a2 a3): a1 = NoV k + 1 - k, a2 = NoL k + 1 - k, a3 = 1 - r2 + 4 pi r2
      const float gv = -(gnv * nv);             // dLoss/dlog a_i
      const float g1 = gv * ia1, g2 = gv * ia2;
      gr2 = gr2 + (gv * ia3) * (c3 - 1.0f) + 0.5f * (g1 * (NoV - 1.0f) + g2 * (NoL - 1.0f));
      gnov = gnov + g1 * k;
      if (cosv > EPS) gcos = gcos + g2 * k;
      q.n = vadd(q.n, vsmul(gcos, L));
    }
    light(l, gi);
  }
  if (nov > EPS) q.n = vadd(q.n, vsmul(gnov, V));
  // f0 = m a + (1 - m) d0
  q.m = vdot(gf0, v3(a.x - d0, a.y - d0, a.z - d0));
  q.a = vadd(q.a, vsmul(m, gf0));
  q.r = r_free ? gr2 * (2.0f * r) : 0.0f;
  return q;
}

// Weights, position and interpolated inputs of pixel (px, py) on face f.
struct DiffFrag {
  float w[3];
  int vi[3];
  V3 pos, nraw, a;
  float r, m;
};

__device__ __forceinline__ void diff_fragment(const DiffArgs& A, uint32_t f, int px, int py, DiffFrag& q) {
  ShadeArgs s;  // only the camera and positions are read by fragment()
  s.cam = A.cam;
  s.mesh.verts = A.soup;
  s.mesh.norms = 0;
  s.mesh.coors = 0;
  s.mesh.colors = 0;
  s.flags = 0;
  Frag fr;
  fragment(s, f, px, py, fr);
  q.w[0] = fr.w0;
  q.w[1] = fr.w1;
  q.w[2] = fr.w2;
  q.pos = fr.pos;
  const int* fc = (const int*)gptr(A.faces) + 3 * (size_t)f;
  gf32* nrm = gptr(A.nrm);
  gf32* col = gptr(A.col);
  gf32* rgh = gptr(A.rough);
  gf32* mtl = gptr(A.metal);
  q.nraw = vs(0.0f);
  q.a = vs(0.0f);
  q.r = 0.0f;
  q.m = 0.0f;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int v = fc[k];
    q.vi[k] = v;
    q.nraw = vadd(q.nraw, vsmul(q.w[k], ld3(nrm + 3 * (size_t)v)));
    q.a = vadd(q.a, vsmul(q.w[k], ld3(col + 3 * (size_t)v)));
    q.r = q.r + q.w[k] * rgh[v];
    q.m = q.m + q.w[k] * mtl[v];
  }
}

__global__ void __launch_bounds__(kBlock)
k_dshade_fwd(const DiffArgs A, const uint64_t* __restrict__ keys, float* __restrict__ img) {
  const long npix = (long)A.cam.W * A.cam.H;
  const long P = (long)blockIdx.x * kBlock + threadIdx.x;
  if (P >= npix) return;
  const uint64_t key = keys[P];
  V3 c = vs(0.0f);
  const uint32_t f = (uint32_t)key - A.id_base;
  if (key_depth(key) < TINA_MAXDEPTH && f < (uint32_t)A.nfaces) {
    const int px = (int)(P % A.cam.W), py = (int)(P / A.cam.W);
    DiffFrag q;
    diff_fragment(A, f, px, py, q);
    const V3 n = vnormalized(q.nraw);
    const V3 V = vneg(view_ray(A.cam, px, py));
    c = diff_color(A, gptr(A.inten), q.a, n, q.r, q.m, q.pos, V);
  } else if (key_depth(key) < TINA_MAXDEPTH) {
    return;  // another object's pixel
  }
  store_rgb(img, P, c);
}

// What bounded the adjoint was not its arithmetic but its atomics: 24 float adds a
// pixel to the three vertices, and one a wave and light to the same few intensity
// words (each about 40 ns behind the last).  A workgroup now takes 16 x 16 pixels
// at a time and adds them up in LDS, in a hash table of vertices (512 slots; a
// vertex that finds no slot in 16 probes goes straight to memory) that is
// flushed with eight adds a vertex, and keeps the intensity sums until it ends.
// The hand-written adjoint takes a third of the arithmetic of the eight-way
// forward-mode duals before it and no scratch.  1024 x 1024, 101 k vertices, 3
// lights: 911 -> 117 us; eight workgroups a CU (two rounds, dealt as they finish)
// against two / three / four: a fit step of 236 us against 275 / 267 / 266.
constexpr int kDiffTile = 16;
constexpr long kDiffGridPerCu = 8;
constexpr int kDiffSlots = 512, kDiffProbes = 16;
static_assert(kDiffTile * kDiffTile == kBlock, "a lane a pixel");

__global__ void __launch_bounds__(kBlock)
k_dshade_bwd(const DiffArgs A, const uint64_t* __restrict__ keys, const float* __restrict__ gimg,
             float* __restrict__ g_col, float* __restrict__ g_nrm, float* __restrict__ g_rough,
             float* __restrict__ g_metal, float* __restrict__ g_inten) {
  __shared__ int s_vert[kDiffSlots];            // vertex of each slot, -1: free
  __shared__ float s_g[8][kDiffSlots];          // its gradient: albedo, normal, roughness, metallic
  __shared__ float s_inten[TINA_MAX_LIGHTS];
  const int tid = threadIdx.x;
  const int tiles_x = (A.cam.W + kDiffTile - 1) / kDiffTile;
  const int ntiles = tiles_x * ((A.cam.H + kDiffTile - 1) / kDiffTile);
  if (tid < TINA_MAX_LIGHTS) s_inten[tid] = 0.0f;
  for (int i = tid; i < kDiffSlots; i += kBlock) {
    s_vert[i] = -1;
#pragma unroll
    for (int c = 0; c < 8; c++) s_g[c][i] = 0.0f;
  }
  __syncthreads();
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int px = (t % tiles_x) * kDiffTile + tid % kDiffTile, py = (t / tiles_x) * kDiffTile + tid / kDiffTile;
    const long P = (long)py * A.cam.W + px;
    bool live = false;
    uint32_t f = 0;
    if (px < A.cam.W && py < A.cam.H) {
      const uint64_t key = keys[P];
      f = (uint32_t)key - A.id_base;
      live = key_depth(key) < TINA_MAXDEPTH && f < (uint32_t)A.nfaces;
    }
    if (__any(live)) {
      DiffFrag q;
      V3 g = vs(0.0f), n = vs(0.0f), V = vs(0.0f);
      float inv = 0.0f;
      q.a = q.pos = vs(0.0f);
      q.r = q.m = 0.0f;
      if (live) {
        g = ld3(gimg + 3 * P);
        diff_fragment(A, f, px, py, q);
        inv = fdiv_rn(1.0f, sqrtf(vdot(q.nraw, q.nraw)));
        n = vsmul(inv, q.nraw);
        V = vneg(view_ray(A.cam, px, py));
      }
      const DiffGrad d = diff_adjoint(A, gptr(A.inten), q.a, n, q.r, q.m, q.pos, V, g, live, [&](int l, float gi) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) gi += __shfl_xor(gi, o);
        if (__lane_id() == 0 && gi != 0.0f) atomicAdd(&s_inten[l], gi);
      });
      if (live) {
        // d n / d nraw = (I - n n^T) / |nraw|
        const V3 graw = vsmul(inv, vsub(d.n, vsmul(vdot(n, d.n), n)));
        const float v[8] = {d.a.x, d.a.y, d.a.z, graw.x, graw.y, graw.z, d.r, d.m};
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const int vi = q.vi[k];
          uint32_t s = ((uint32_t)vi * 0x9e3779b1u) >> (32 - 9);
          int at = -1;
#pragma unroll 1
          for (int p = 0; p < kDiffProbes; p++) {
            const int had = atomicCAS(&s_vert[s], -1, vi);
            if (had == -1 || had == vi) {
              at = (int)s;
              break;
            }
            s = (s + 1) % kDiffSlots;
          }
          if (at >= 0) {
#pragma unroll
            for (int c = 0; c < 8; c++) atomicAdd(&s_g[c][at], q.w[k] * v[c]);
          } else {                               // a crowded table: straight to memory
#pragma unroll
            for (int c = 0; c < 3; c++) {
              atomicAdd(g_col + 3 * (size_t)vi + c, q.w[k] * v[c]);
              atomicAdd(g_nrm + 3 * (size_t)vi + c, q.w[k] * v[3 + c]);
            }
            atomicAdd(g_rough + vi, q.w[k] * v[6]);
            atomicAdd(g_metal + vi, q.w[k] * v[7]);
          }
        }
      }
    }
    __syncthreads();
    for (int i = tid; i < kDiffSlots; i += kBlock) {
      const int vi = s_vert[i];
      if (vi < 0) continue;
      s_vert[i] = -1;
      float v[8];
#pragma unroll
      for (int c = 0; c < 8; c++) {
        v[c] = s_g[c][i];
        s_g[c][i] = 0.0f;
      }
#pragma unroll
      for (int c = 0; c < 3; c++) {
        atomicAdd(g_col + 3 * (size_t)vi + c, v[c]);
        atomicAdd(g_nrm + 3 * (size_t)vi + c, v[3 + c]);
      }
      atomicAdd(g_rough + vi, v[6]);
      atomicAdd(g_metal + vi, v[7]);
    }
    __syncthreads();
  }
  if (tid < A.nlights && s_inten[tid] != 0.0f) atomicAdd(g_inten + tid, s_inten[tid]);
}

}  // namespace tina
