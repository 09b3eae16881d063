// ssr_kernels.h -- screen-space reflections (tina/postp/ssr.py:6-103).
//
//   k_depth_span nearest and farthest depth of every block of pixels
//   k_ssr        SSR.render_at for the pixels one object won: the view position
//                from the depth buffer, nsamples directions drawn from the
//                object's material (IMaterial.sample, material.py:25-32,
//                124-138, 181-184, 228-238, 365-384, 398-405, 467-477), each
//                marched nsteps steps through the depth buffer; a step landing
//                within the tolerance behind the depth there takes the image
//                colour at that point times the sample weight.
//   k_ssr_apply  SSR.apply: the blur x blur box mean of the reflection buffer
//                (at offset -blur / 2), image * (1 - a) + rgb.
//
// The random stream is the reference's WangHashRNG (tina/random.py:17-64)
// seeded with the pixel's position modulo the box size, so the non-TAA mode
// draws the reference's own numbers.  cos and sin are evaluated in binary64 and
// rounded (the reference's ti.cos / ti.sin codegen is not pinned); every other
// expression keeps the reference's grouping.  Reads past the screen clamp to
// it (the reference reads outside its fields there).
#pragma once
#include "postp_kernels.h"

namespace tina {

// WangHashRNG._noise (random.py:28-35), in uint32 arithmetic
__device__ __forceinline__ uint32_t wang_noise(uint32_t v) {
  v = (v ^ 61u) ^ (v >> 16);
  v *= 9u;
  v ^= v << 4;
  v *= 0x27d4eb2du;
  v ^= v >> 15;
  return v;
}

struct WangRNG {
  uint32_t seed;
  // random(): noise_int(seed) >> 1, times 2 / 2^32 (random.py:38-41, 54-57)
  __device__ __forceinline__ float random() {
    const uint32_t u = wang_noise(seed) >> 1;
    seed += 1u;
    return (float)u * 4.656612873077393e-10f;
  }
  __device__ __forceinline__ uint32_t random_int() {
    const uint32_t u = wang_noise(seed);
    seed += 1u;
    return u;
  }
};

// cos and sin of a binary32 angle in [0, 2 pi], in binary64 and rounded: the
// multiple of pi / 2 taken off in two parts, then the Taylor series to x^16
// (the next term is below 2^-53 of the result on [-pi / 4, pi / 4]).
__device__ __forceinline__ void azimuth(float a, float& c, float& s) {
  const double x = (double)a, q = rint(x * 0.63661977236758134);
  const double r = __builtin_fma(-q, 6.123233995736766e-17, __builtin_fma(-q, 1.5707963267948966, x)), z = r * r;
  double ps = -7.647163731819816e-13, pc = 4.779477332387385e-14;  // -1 / 15!, 1 / 16!
  ps = __builtin_fma(ps, z, 1.6059043836821613e-10);
  pc = __builtin_fma(pc, z, -1.1470745597729725e-11);
  ps = __builtin_fma(ps, z, -2.5052108385441720e-08);
  pc = __builtin_fma(pc, z, 2.0876756987868100e-09);
  ps = __builtin_fma(ps, z, 2.7557319223985893e-06);
  pc = __builtin_fma(pc, z, -2.7557319223985888e-07);
  ps = __builtin_fma(ps, z, -1.9841269841269841e-04);
  pc = __builtin_fma(pc, z, 2.4801587301587302e-05);
  ps = __builtin_fma(ps, z, 8.3333333333333332e-03);
  pc = __builtin_fma(pc, z, -1.3888888888888889e-03);
  ps = __builtin_fma(ps, z, -1.6666666666666666e-01);
  pc = __builtin_fma(pc, z, 4.1666666666666664e-02);
  pc = __builtin_fma(pc, z, -0.5);
  const float sr = (float)__builtin_fma(ps * z, r, r), cr = (float)__builtin_fma(pc, z, 1.0);
  const int n = (int)q;
  const float s0 = n & 1 ? cr : sr, c0 = n & 1 ? sr : cr;
  s = n & 2 ? -s0 : s0;
  c = (n + 1) & 2 ? -c0 : c0;
}

// spherical(h, p) (tina/advans.py:105-108): (sqrt(max(0, 1 - h^2)) (cos, sin)(p tau), h)
__device__ __forceinline__ V3 spherical(float h, float p) {
  float c, s;
  azimuth(p * 6.2831855f, c, s);
  const float r = sqrtf(fmaxf(0.0f, 1.0f - h * h));
  return v3(r * c, r * s, h);
}

// tangentspace(n) (advans.py:97-100): columns tan, bitan, n
struct Tangent {
  V3 tan, bitan, n;
};
__device__ __forceinline__ Tangent tangent_space(V3 n) {
  Tangent t;
  t.bitan = vnormalized(vcross(n, v3(233.0f, 666.0f, 512.0f)));
  t.tan = vcross(t.bitan, n);
  t.n = n;
  return t;
}
// tangentspace @ d
__device__ __forceinline__ V3 tangent_apply(const Tangent& t, V3 d) {
  return v3(((t.tan.x * d.x) + (t.bitan.x * d.y)) + (t.n.x * d.z), ((t.tan.y * d.x) + (t.bitan.y * d.y)) + (t.n.y * d.z),
            ((t.tan.z * d.x) + (t.bitan.z * d.y)) + (t.n.z * d.z));
}
__device__ __forceinline__ V3 tangent_apply(V3 n, V3 d) { return tangent_apply(tangent_space(n), d); }

// CookTorrance.sub_brdf (material.py:323-357): the Fresnel and visibility terms
__device__ __forceinline__ void ct_sub(float roughness, V3 f0, V3 n, V3 L, V3 V, V3& fdf, float& vdf) {
  const float EPS = 1e-10f;
  const float ONE_M_EPS = (float)(1.0 - 1e-10);
  const V3 half = vnormalized(vadd(L, V));
  const float NoL = fmaxf(EPS, vdot(L, n));
  const float NoV = fmaxf(EPS, vdot(V, n));
  const float VoH = fminf(ONE_M_EPS, fmaxf(EPS, vdot(half, V)));
  const float alpha2 = fmaxf(1e-6f, roughness * roughness);
  const float k = alpha2 * 0.5f;  // x * 0.5 is x / 2 to the bit
  vdf = fdiv_rn(1.0f, ((NoV * k) + 1.0f) - k);
  vdf = vdf * fdiv_rn(1.0f, ((NoL * k) + 1.0f) - k);
  vdf = fdiv_rn(vdf, (1.0f * (1.0f - alpha2)) + ((float)(4.0 * 3.141592653589793) * alpha2));
  const float x1 = 1.0f - VoH, x2 = x1 * x1;
  const float p5 = (x2 * x2) * x1;
  fdf = vadd(f0, vsmul(p5, vsub(vs(1.0f), f0)));
}

// MixMaterial.sample (material.py:124-138) of a pixel with mix factor fac: the
// chance f of the second material and the factors its and the first's weights take.
struct MixDraw {
  float f;
  V3 first, second;
};
__device__ __forceinline__ MixDraw mix_draw(V3 fac, bool scalar) {
  MixDraw x;
  float f = scalar ? fac.x : fdiv_rn((fac.x + fac.y) + fac.z, 3.0f);   // Vavg
  if (f != 0.0f && f != 1.0f) {              // smoothlerp(f, 0.12, 0.88)
    const float t = fminf(1.0f, fmaxf(0.0f, f));
    const float s = (t * t) * (3.0f - 2.0f * t);
    f = 0.12f * (1.0f - s) + 0.88f * s;
  }
  x.f = f;
  x.second = scalar ? vs(fdiv_rn(fac.x, f)) : vdivs(fac, f);
  x.first = scalar ? vs(fdiv_rn(1.0f - fac.x, 1.0f - f)) : vdivs(vsub(vs(1.0f), fac), 1.0f - f);
  return x;
}

// One draw of material.sample(idir, nrm, 1, rng) for the program m: the
// combinators pick a branch (MixMaterial with probability smoothlerp(avg(fac),
// .12, .88), AddMaterial by a random integer's parity), the leaf samples its
// lobe, and the branch factors multiply the leaf's weight innermost first.
__device__ __forceinline__ void material_sample(const tina_material& m, const Slots& pv, V3 idir, V3 nrm,
                                                WangRNG& rng, V3& odir, V3& wei) {
  int size[TINA_MAX_OPS];
  for (int i = 0; i < m.nops; i++) {
    const tina_op o = op_at(m, i);
    if (o.op <= TINA_OP_EMISSION) size[i] = 1;
    else if (o.op == TINA_OP_SCALE) size[i] = 1 + size[i - 1];
    else size[i] = 1 + size[i - 1] + size[i - 1 - size[i - 1]];
  }
  V3 fac_stack[TINA_MAX_OPS];
  int nfac = 0;
  int node = m.nops - 1;
  for (;;) {
    const tina_op o = op_at(m, node);
    if (o.op <= TINA_OP_EMISSION) break;
    if (o.op == TINA_OP_SCALE) {             // ScaleMaterial.sample: wei * fac
      fac_stack[nfac++] = pv.get(o.a);
      node = node - 1;
    } else if (o.op == TINA_OP_MIX) {        // MixMaterial.sample (material.py:124-138)
      const MixDraw x = mix_draw(pv.get(o.a), param_at(m, o.a).dim == 1);
      if (rng.random() < x.f) {
        fac_stack[nfac++] = x.second;
        node = node - 1;
      } else {
        fac_stack[nfac++] = x.first;
        node = node - 1 - size[node - 1];
      }
    } else {                                 // AddMaterial.sample (material.py:228-238)
      const bool first = (rng.random_int() % 2u) == 0u;
      fac_stack[nfac++] = vs(2.0f);
      node = first ? node - 1 - size[node - 1] : node - 1;
    }
  }
  const tina_op leaf = op_at(m, node);
  wei = vs(0.0f);
  odir = idir;
  if (leaf.op == TINA_OP_LAMBERT) {          // Lambert.sample (material.py:398-405)
    float u = rng.random();
    const float v = rng.random();
    u = sqrtf(u);
    odir = vnormalized(tangent_apply(nrm, spherical(u, v)));
    wei = vs(1.0f);
  } else if (leaf.op == TINA_OP_COOKTORRANCE) {  // CookTorrance.sample (material.py:365-384)
    const float roughness = pv.get(leaf.a).x;
    const V3 f0 = pv.get(leaf.b);
    const float alpha2 = fmaxf(0.0f, roughness * roughness);
    float u = rng.random();
    const float v = rng.random();
    u = sqrtf(fdiv_rn(1.0f - u, 1.0f - u * (1.0f - alpha2)));
    const V3 rdir = vreflect(vneg(idir), nrm);
    odir = tangent_apply(rdir, spherical(u, v));
    V3 fdf;
    float vdf;
    ct_sub(roughness, f0, nrm, idir, odir, fdf, vdf);
    if (vdot(odir, nrm) < 0.0f) {
      odir = vneg(odir);
      fdf = vs(0.0f);
    }
    wei = vsmul(vdf, fdf);
  } else if (leaf.op == TINA_OP_PHONG || leaf.op == TINA_OP_BLINNPHONG) {
    // Phong.sample (material.py:467-477); the Blinn-Phong lobe (an extension with
    // no sample of its own) draws the same directions
    const float mm = pv.get(leaf.a).x;
    float u = rng.random();
    const float v = rng.random();
    u = (float)pow((double)u, (double)fdiv_rn(1.0f, mm + 1.0f));
    const V3 rdir = vreflect(vneg(idir), nrm);
    odir = tangent_apply(rdir, spherical(u, v));
    float w = 1.0f;
    if (vdot(odir, nrm) < 0.0f) {
      odir = vneg(odir);
      w = 0.0f;
    }
    wei = vs(w);
  }  // Emission.sample: (idir, 0, 0)
  for (int i = nfac - 1; i >= 0; i--) wei = vmul(wei, fac_stack[i]);
}

// mapply_pos for a march step, with the range test on the divisor alone: as
// mapply_pos to the bit wherever a component lies between 2^-50 and 1 in magnitude,
// outside [-1, 1] or NaN where that is.  The quotient's two corrections are exact as
// long as their remainders are no subnormals, for numerators down to 2^-110.  A smaller
// one over a divisor of at least 2^-60 gives a quotient below 2^-50, which may differ in
// its last bit: added to 0.5 for the pixel, or compared with depths a multiple of 2^-30
// apart, it is the same.  A numerator above the shared division's range, or infinite,
// gives a quotient outside [-1, 1] or a NaN.
__device__ __forceinline__ V3 march_project(const float* __restrict__ M, V3 p) {
  float r0, r1, r2, w;
  mapply1(M, p.x, p.y, p.z, r0, r1, r2, w);
  const RcpRN R = rcp_rn(w);
  if (!R.ok) return v3(r0 / w, r1 / w, r2 / w);
  auto quo = [&](float a) {
    const float q = a * R.r;
    const float q3 = __builtin_fmaf(__builtin_fmaf(-R.d, q, a), R.r, q);
    return __builtin_fmaf(__builtin_fmaf(-R.d, q3, a), R.r, q3);
  };
  return v3(quo(r0), quo(r1), quo(r2));
}

// ---- the coarse depth table ----
//
// One word per 2^log x 2^log block of pixels: 1 - depth of its nearest and
// farthest key as two halves, widened so that comparing 1 - z in binary32 with
// them never misses a hit.  A perspective depth sits close below 1, so 1 - depth
// keeps the bits that tell surfaces apart.
constexpr int kSpanWords = 2048;             // at most 8 KB of a workgroup's LDS

inline int span_log(int W, int H) {
  int l = 4;
  while ((long)((W + (1 << l) - 1) >> l) * ((H + (1 << l) - 1) >> l) > kSpanWords) l++;
  return l;
}
inline long span_words(int W, int H) {
  const int l = span_log(W, H);
  return (long)((W + (1 << l) - 1) >> l) * ((H + (1 << l) - 1) >> l);
}

typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

// One wave a block.  The margins cover the halves' rounding (2^-11 of the value)
// and that of 1 - z and 1 - (z - tolerance) (2^-24 each of at most 2).
__global__ void __launch_bounds__(kBlock)
k_depth_span(const uint64_t* __restrict__ keys, int W, int H, int log, uint32_t* __restrict__ span) {
  const int tw = (W + (1 << log) - 1) >> log, n = tw * ((H + (1 << log) - 1) >> log);
  const int b = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (b >= n) return;
  const int x0 = (b % tw) << log, y0 = (b / tw) << log;
  float near = -4.0f, far = 4.0f;
  for (int i = lane; i < 1 << (2 * log); i += 64) {
    const int x = x0 + (i & ((1 << log) - 1)), y = y0 + (i >> log);
    if (x >= W || y >= H) continue;
    const float d = 1.0f - (float)key_depth(keys[(long)y * W + x]) * 0x1p-30f;
    near = fmaxf(near, d);
    far = fminf(far, d);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    near = fmaxf(near, __shfl_xor(near, o));
    far = fminf(far, __shfl_xor(far, o));
  }
  if (lane == 0) {
    const h16x2 h = {(_Float16)(near + (1e-6f + fabsf(near) * 1e-3f)), (_Float16)(far - (1e-6f + fabsf(far) * 1e-3f))};
    span[b] = __builtin_bit_cast(uint32_t, h);
  }
}

// The SSR arguments: the object's mesh and material and the camera (ShadeArgs),
// the screen buffers and the march parameters.
struct SsrArgs {
  const float* norm;   // [H][W][3] NormalShader buffer
  const float* coor;   // [H][W][2] TexcoordShader buffer, or null (texcoord 0)
  const float* image;  // [H][W][3] the linear image the reflections sample
  float* out;          // [H][W][4] rgb + hit fraction
  int nsamples, nsteps, blur, taa;
  float stepsize, tolerance;
  const uint32_t* span;  // the coarse depth table of the keys
  int span_log;
  uint32_t seed;       // the TAA mode's frame seed
};

// A pixel's draws from its object's material.  The fixed programs (Diffuse,
// Classic, Blinn, PBR) work out once what does not change between draws: the two
// tangent frames, the mix chance and factors.  A draw picks its frame by address, so
// under Classic, Blinn and PBR the compiler keeps them in scratch (164 bytes a lane,
// read back by every sample); picked by component they stay in registers, at a wave a
// SIMD less: 1,351 us for the effects frame below instead of 1,264.  Any other tree
// walks its program (material_sample, whose stacks live in scratch).
template <int PROG>
struct SsrDraw {
  static constexpr int kDraws = PROG == PROG_DIFFUSE ? 2 : 3;  // numbers a sample takes from the stream
  V3 V, nrm, f0;
  Tangent tn, tr;          // about the normal and about the mirrored view direction
  MixDraw mix;
  V3 lam;                  // the Lambert side's weight
  float lobe, alpha2, inv_m;  // roughness or shininess; max(0, r^2); 1 / (m + 1)

  __device__ __forceinline__ void init(const tina_material& m, uint32_t f, const Frag& fr, V3 viewdir) {
    V = viewdir;
    nrm = fr.nrm;
    tn = tangent_space(nrm);
    lam = eval_slot(m, m.ops[1].a, f, fr);
    if constexpr (PROG != PROG_DIFFUSE) {
      mix = mix_draw(eval_slot(m, m.ops[3].a, f, fr), param_at(m, m.ops[3].a).dim == 1);
      lam = vmul(lam, mix.first);
      tr = tangent_space(vreflect(vneg(V), nrm));
      lobe = eval_slot(m, m.ops[2].a, f, fr).x;
      if constexpr (PROG == PROG_PBR) {
        f0 = eval_slot(m, m.ops[2].b, f, fr);
        alpha2 = fmaxf(0.0f, lobe * lobe);
      } else {
        inv_m = fdiv_rn(1.0f, lobe + 1.0f);
      }
    }
  }

  // the draws and expressions of material_sample for the same program
  __device__ __forceinline__ void sample(const tina_material&, WangRNG& rng, V3& odir, V3& wei) const {
    const bool diff = PROG == PROG_DIFFUSE || !(rng.random() < mix.f);
    float u = rng.random();
    const float v = rng.random();
    if (PROG == PROG_PBR || PROG == PROG_DIFFUSE) {
      if (!diff) u = fdiv_rn(1.0f - u, 1.0f - u * (1.0f - alpha2));
      u = sqrtf(u);
    } else {
      u = diff ? sqrtf(u) : (float)pow((double)u, (double)inv_m);
    }
    odir = tangent_apply(diff ? tn : tr, spherical(u, v));
    if (diff) {
      odir = vnormalized(odir);
      wei = lam;
    } else if (PROG == PROG_PBR) {
      V3 fdf;
      float vdf;
      ct_sub(lobe, f0, nrm, V, odir, fdf, vdf);
      if (vdot(odir, nrm) < 0.0f) {
        odir = vneg(odir);
        fdf = vs(0.0f);
      }
      wei = vmul(vsmul(vdf, fdf), mix.second);
    } else {
      float w = 1.0f;
      if (vdot(odir, nrm) < 0.0f) {
        odir = vneg(odir);
        w = 0.0f;
      }
      wei = vmul(vs(w), mix.second);
    }
  }
};

template <>
struct SsrDraw<PROG_GENERIC> {
  V3 V, nrm;
  Slots pv;
  __device__ __forceinline__ void init(const tina_material& m, uint32_t f, const Frag& fr, V3 viewdir) {
    V = viewdir;
    nrm = fr.nrm;
    eval_params(m, f, fr.pos, fr.nrm, fr.tc, fr.color, pv);
  }
  __device__ __forceinline__ void sample(const tina_material& m, WangRNG& rng, V3& odir, V3& wei) const {
    material_sample(m, pv, V, nrm, rng, odir, wei);
  }
};

// A wave takes an 8 x 8 block of pixels, so its rays start side by side; a
// workgroup's kSsrSlices waves share the block's pixels and split their samples
// (a fixed program draws the same count of numbers every sample, so a run's
// stream can start anywhere).  One wave a block of pixels left an object of 125 k
// pixels with two waves a SIMD.
//
// What bounds the march: VALU issue -- a projection with three correctly rounded
// quotients a step, about 88 instructions -- once the key reads are out of the
// way.  The 7.4 MB of keys of a 1279 x 721 frame do not fit an XCD's L2 and a
// wave's rays touch a line each, so a step first asks the coarse depth table in
// LDS whether a surface of its block of pixels can be in reach, and reads the key
// only then (143 M L2 requests of one pass became 16 M).  A lane marches two
// steps at a time with both reads in flight and takes its ray's colour once the
// wave's rays have all ended, not where each ends.  Giving a lane its next sample
// while others still march (from 16, 32 or 48 waiting lanes on) cost 4-6 % more in
// repeated sampling than the idle lanes do.
//
// A 1279 x 721 frame with every effect on, two PBR objects over 433 k pixels, 32
// samples x 32 steps: 4,295 us with a pixel a lane and the material walked, with
// binary64 cos and sin calls, every sample; 2,249 with the fixed programs; 1,674
// with four slices (8: 1,753, 16: 2,046); 1,281 with the coarse table.  Its blocks
// of 16 pixels instead of 32 (in 32 KB) gain 1 % and cost the LDS of two workgroups.
constexpr int kSsrTile = 8;
constexpr int kSsrSlices = 4;
constexpr int kSsrRun = 8;                   // samples a slice traces a round

template <int PROG, int SLICES>
__global__ void __launch_bounds__(64 * SLICES)
k_ssr(const ShadeArgs a_by_value, const uint64_t* __restrict__ keys, const SsrArgs s) {
  (void)a_by_value;
#if defined(__HIP_DEVICE_COMPILE__)
  const ShadeArgs& a = *(const ShadeArgs*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  const ShadeArgs& a = a_by_value;
#endif
  const Cam& cam = a.cam;
  const float resx = (float)cam.W, resy = (float)cam.H;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tiles_x = (cam.W + kSsrTile - 1) / kSsrTile;
  const int x = (int)(blockIdx.x % tiles_x) * kSsrTile + lane % kSsrTile;
  const int y = (int)(blockIdx.x / tiles_x) * kSsrTile + lane / kSsrTile;
  const long P = (long)y * cam.W + x;
  uint64_t k = empty_key();
  if (x < cam.W && y < cam.H) k = keys[P];
  const uint32_t f = (uint32_t)k - a.mesh.id_base;
  float* o = s.out + 4 * P;
  bool live = key_depth(k) < TINA_MAXDEPTH && f < (uint32_t)a.mesh.nfaces;
  Frag fr;
  fr.nrm = vs(0.0f);
  if (live) {
    fr.nrm = ld_px(s.norm, cam.W, x, y);
    if (vdot(fr.nrm, fr.nrm) < 1e-6f) {      // norm_sqr() < eps: nothing to reflect
      if (wave == 0) o[0] = o[1] = o[2] = o[3] = 0.0f;
      live = false;
    }
  }
  if (!__any(live)) return;                  // the same for every wave: they hold the same pixels
  extern __shared__ __align__(16) uint32_t s_span[];
  const int slog = s.span_log, span_w = (cam.W + (1 << slog) - 1) >> slog;
  const int nspan = span_w * ((cam.H + (1 << slog) - 1) >> slog);
  for (int i = threadIdx.x; i < nspan; i += 64 * SLICES) s_span[i] = s.span[i];
  __syncthreads();
  SsrDraw<PROG> draw;
  WangRNG rng;
  const float nst = (float)s.nsteps;
  float vtol = 0.0f;
  if (live) {
    fr.tc = s.coor ? v3(s.coor[2 * P], s.coor[2 * P + 1], 0.0f) : vs(0.0f);
    fr.color = vs(1.0f);                     // Input('color') is (1, 1, 1) here
    const float p_x = (float)x + cam.bias[0], p_y = (float)y + cam.bias[1];
    const V3 vpos = v3((fdiv_rn(p_x, resx) * 2.0f) - 1.0f, (fdiv_rn(p_y, resy) * 2.0f) - 1.0f,
                       (float)key_depth(k) * 0x1p-30f);
    fr.pos = mapply_pos(cam.V2W, vpos);
    const V3 viewdir = vneg(view_ray(cam, x, y));
    draw.init(a.mat, f, fr, viewdir);
    if (!s.taa) {
      // WangHashRNG(P % blurring): noise_int of the 2-vector (random.py:43-52)
      rng.seed = wang_noise((uint32_t)(y % s.blur) ^ wang_noise((uint32_t)(x % s.blur)));
    } else {
      rng.seed = wang_noise((uint32_t)y ^ wang_noise((uint32_t)x ^ wang_noise(s.seed)));
    }
    const V3 vpz = mapply_pos(cam.W2V, fr.pos);
    vtol = s.tolerance * (mapply_pos(cam.W2V, vsub(fr.pos, v3(fdiv_rn(viewdir.x, nst), fdiv_rn(viewdir.y, nst),
                                                              fdiv_rn(viewdir.z, nst)))).z - vpz.z);
  }
  const uint32_t* __restrict__ khi = (const uint32_t*)keys + 1;  // the depth half of a key
  const float xmax = (float)(cam.W - 1), ymax = (float)(cam.H - 1);
  float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f, r3 = 0.0f;
  // one sample: the colour its ray meets times its weight, 0 when it meets nothing
  auto trace = [&](V3& clr) {
    V3 odir, wei;
    draw.sample(a.mat, rng, odir, wei);
    const float c = vdot(odir, draw.V);
    const float step = fdiv_rn(s.stepsize, sqrtf(1.0f - c * c) * nst);
    const float jit = rng.random();
    V3 ro = vadd(fr.pos, vsmul(step, vsmul(jit, odir)));
    const V3 sd = vsmul(step, odir);
    bool hit = false;                          // the ray ended on a surface, at (hx, hy)
    float hx = 0.0f, hy = 0.0f;
    for (int j = s.nsteps; j > 0;) {
      V3 vro[2];
      float Dx[2], Dy[2];
      uint32_t kd[2] = {0u, 0u};
      bool in[2], near[2];                     // on the screen; in reach of a surface of its block
#pragma unroll
      for (int t = 0; t < 2; t++) {
        ro = vadd(ro, sd);
        vro[t] = march_project(cam.W2V, ro);
        in[t] = (fabsf(vro[t].x) <= 1.0f) & (fabsf(vro[t].y) <= 1.0f) & (fabsf(vro[t].z) <= 1.0f);
        Dx[t] = (vro[t].x * 0.5f + 0.5f) * resx;
        Dy[t] = (vro[t].y * 0.5f + 0.5f) * resy;
        // on the screen for any value (a NaN is 0); the reference's own pixel when `in`
        const uint32_t ix = (uint32_t)fminf(fmaxf(Dx[t], 0.0f), xmax), iy = (uint32_t)fminf(fmaxf(Dy[t], 0.0f), ymax);
        const h16x2 h = __builtin_bit_cast(h16x2, s_span[(iy >> slog) * (uint32_t)span_w + (ix >> slog)]);
        // not in front of the block's nearest surface, nor beyond the tolerance of its farthest
        near[t] = in[t] & !(1.0f - vro[t].z >= (float)h[0]) & !(1.0f - (vro[t].z - vtol) <= (float)h[1]);
        if (near[t]) kd[t] = *(const uint32_t*)((const char*)khi + 8ull * (iy * (uint32_t)cam.W + ix));
      }
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const float depth = (float)(int32_t)(kd[t] ^ 0x80000000u) * 0x1p-30f;
        const bool meets = near[t] & (vro[t].z - vtol < depth) & (depth < vro[t].z);
        if (j > 0) {
          j = (in[t] && !meets) ? j - 1 : 0;
          hit = meets;
          hx = Dx[t];
          hy = Dy[t];
        }
      }
    }
    clr = vs(0.0f);
    if (hit) {
      clr = vmul(bilerp_img(s.image, cam.W, cam.H, hx, hy), wei);
      r3 = r3 + 1.0f;
    }
  };
  if constexpr (SLICES == 1) {
    for (int i = live ? 0 : s.nsamples; i < s.nsamples; i++) {
      V3 clr;
      trace(clr);
      r0 = r0 + clr.x;
      r1 = r1 + clr.y;
      r2 = r2 + clr.z;
    }
  } else {
    // rounds of SLICES runs of `per` samples; the first slice adds the round's
    // colours in sample order (FXAA branches on the image: the sums keep their bits)
    __shared__ float s_c[(SLICES - 1) * kSsrRun][3][64], s_n[SLICES][64];
    const uint32_t seed0 = rng.seed;
    const int ns = s.nsamples, per = min(kSsrRun, (ns + SLICES - 1) / SLICES);
    for (int base = 0; base < ns; base += SLICES * per) {
      const int first = base + wave * per;
      rng.seed = seed0 + (uint32_t)(SsrDraw<PROG>::kDraws + 1) * (uint32_t)first;
      for (int i = 0; live && i < per && first + i < ns; i++) {
        V3 clr;
        trace(clr);
        if (wave == 0) {
          r0 = r0 + clr.x;
          r1 = r1 + clr.y;
          r2 = r2 + clr.z;
        } else {
          float(*q)[64] = s_c[(wave - 1) * per + i];
          q[0][lane] = clr.x;
          q[1][lane] = clr.y;
          q[2][lane] = clr.z;
        }
      }
      __syncthreads();
      if (wave == 0) {
        const int n = min(ns - base, SLICES * per) - per;
        for (int i = 0; i < n; i++) {
          r0 = r0 + s_c[i][0][lane];
          r1 = r1 + s_c[i][1][lane];
          r2 = r2 + s_c[i][2][lane];
        }
      }
      __syncthreads();
    }
    s_n[wave][lane] = r3;                      // counts: exact in any order
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 1; w < SLICES; w++) r3 = r3 + s_n[w][lane];
  }
  if (live) {
    const float ns = (float)s.nsamples;
    o[0] = fdiv_rn(r0, ns);
    o[1] = fdiv_rn(r1, ns);
    o[2] = fdiv_rn(r2, ns);
    o[3] = fdiv_rn(r3, ns);
  }
}

template <int PROG, int SLICES>
void launch_ssr(int W, int H, hipStream_t st, const ShadeArgs& a, const uint64_t* keys, const SsrArgs& s) {
  const long tiles = (long)((W + kSsrTile - 1) / kSsrTile) * ((H + kSsrTile - 1) / kSsrTile);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ssr<PROG, SLICES>), dim3((unsigned)tiles), dim3(64 * SLICES),
                     (size_t)span_words(W, H) * 4, st, a, keys, s);
}

// A single sample has nothing to split: the waves without one only repeated the
// pixel's set-up (1279 x 721, one object over the screen, frame with Classic 382 us,
// PBR 314, Diffuse 265 with four slices; 235, 236 and 204 with one.  Two samples: 391,
// 331 and 280 against 282, 280 and 246, but 138 against 150 at 320 x 180, where four
// times the waves count for more).
template <int PROG>
void launch_ssr_fixed(int W, int H, hipStream_t st, const ShadeArgs& a, const uint64_t* keys, const SsrArgs& s) {
  if (s.nsamples > 1)
    launch_ssr<PROG, kSsrSlices>(W, H, st, a, keys, s);
  else
    launch_ssr<PROG, 1>(W, H, st, a, keys, s);
}

inline void dispatch_ssr(int prog, int W, int H, hipStream_t st, const ShadeArgs& a, const uint64_t* keys,
                         const SsrArgs& s) {
  const long n = span_words(W, H);
  hipLaunchKernelGGL(k_depth_span, dim3((unsigned)((n + kBlock / 64 - 1) / (kBlock / 64))), dim3(kBlock), 0, st, keys, W,
                     H, s.span_log, const_cast<uint32_t*>(s.span));
  switch (prog) {
    case PROG_DIFFUSE: launch_ssr_fixed<PROG_DIFFUSE>(W, H, st, a, keys, s); break;
    case PROG_CLASSIC:
    case PROG_BLINN:  // Phong.sample serves both lobes
      launch_ssr_fixed<PROG_CLASSIC>(W, H, st, a, keys, s);
      break;
    case PROG_PBR: launch_ssr_fixed<PROG_PBR>(W, H, st, a, keys, s); break;
    default: launch_ssr<PROG_GENERIC, 1>(W, H, st, a, keys, s); break;
  }
}

// SSR.apply (ssr.py:31-45): res = the blur x blur mean of the buffer at offset
// -blur / 2 (reads clamped; the pixel itself in the TAA mode); image *= 1 - res.w;
// image += res.xyz.
__global__ void __launch_bounds__(kBlock)
k_ssr_apply(float* __restrict__ img, const float* __restrict__ buf, int W, int H, int blur, int taa) {
  const long npix = (long)W * H;
  for (long P = (long)blockIdx.x * kBlock + threadIdx.x; P < npix; P += (long)gridDim.x * kBlock) {
    const int x = (int)(P % W), y = (int)(P / W);
    float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f, r3 = 0.0f;
    if (taa) {
      const float* b = buf + 4 * P;
      r0 = b[0]; r1 = b[1]; r2 = b[2]; r3 = b[3];
    } else {
      const int offs = blur / 2;
      for (int k = 0; k < blur; k++)
        for (int l = 0; l < blur; l++) {
          const int xx = min(max(x + k - offs, 0), W - 1), yy = min(max(y + l - offs, 0), H - 1);
          const float* b = buf + 4 * ((long)yy * W + xx);
          r0 = r0 + b[0]; r1 = r1 + b[1]; r2 = r2 + b[2]; r3 = r3 + b[3];
        }
      const float n = (float)(blur * blur);
      r0 = fdiv_rn(r0, n); r1 = fdiv_rn(r1, n); r2 = fdiv_rn(r2, n); r3 = fdiv_rn(r3, n);
    }
    float* p = img + 3 * P;
    const float m = 1.0f - r3;
    p[0] = p[0] * m + r0;
    p[1] = p[1] * m + r1;
    p[2] = p[2] * m + r2;
  }
}

}  // namespace tina
