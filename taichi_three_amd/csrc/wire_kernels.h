// wire_kernels.h -- WireframeRaster (tina/core/wireframe.py:49-95).
//
//   k_wires   the samples draw_line steps along each wire's screen segment
//             (one pixel per step on the major axis, :50-64) enter the depth|id
//             min with the depth interpolated by the 1/w weights of :83-91.
//             A lane sets a wire up, the wave scans the sample counts and walks
//             the samples, one a lane.  Only the samples whose major-axis position
//             can land on the screen are walked (the range is found in binary64
//             with a margin far above the binary32 rounding of a + k i + bias);
//             each walked sample is evaluated and tested exactly as the reference
//             evaluates it.
//   k_wire_bin, k_wire_tile   the same samples, tile by tile of the screen with
//             the keys in LDS, for calls of many wires.
//   k_paint   blend_color with factor 1 (tina/core/shader.py:134-135): the pixels
//             a range of ids won take one colour (the wire colour).
#pragma once
#include "bin_kernels.h"
#include "shade_dev.h"

namespace tina {

// What one wire keeps: viewport start a, step k, 1 / w of the two ends, their
// view-space z, the step count siz of draw_line and the first walked step i0.
struct WSetup {
  float ax, ay, kx, ky, ws0, ws1, Az, Bz;
  int32_t siz, i0;
};

// Steps i in [lo, hi] of a line whose major-axis position a + k i + bias can fall
// in [0, res): bounds in binary64 widened by 2 + 1e-6 of the magnitudes involved.
__device__ __forceinline__ void wire_major_range(float a, float k, float bias, int res, int32_t siz, int32_t& lo,
                                                 int32_t& hi) {
  lo = 0;
  hi = siz;
  if (!(a == a)) return;  // a NaN start comes with siz = 0: the one step is tested as is
  const double ad = a, bd = bias;
  const double err = 2.0 + (fabs(ad) + (double)siz + fabs(bd) + (double)res) * 1e-6;
  double l, h;
  if (k > 0.0f) {
    l = -ad - bd - err;
    h = (double)res - ad - bd + err;
  } else {
    l = ad + bd - (double)res - err;
    h = ad + bd + err;
  }
  l = fmax(l, 0.0);
  h = fmin(h, (double)siz);
  if (!(l <= h)) {
    hi = -1;
    return;
  }
  lo = (int32_t)ceil(l);  // both in [0, siz]
  hi = (int32_t)floor(h);
}

// false when the wire is clipped (wireframe.py:75-78) or no step can reach the screen
__device__ __forceinline__ bool wire_setup(const Cam& cam, gf32* verts, long f, bool clip, WSetup& s,
                                           uint64_t& count) {
  const V3 Al = ld3(verts + 6 * f), Bl = ld3(verts + 6 * f + 3);
  float wA, wB;
  const V3 Av = mapply_pos(cam.W2V, Al, &wA);
  const V3 Bv = mapply_pos(cam.W2V, Bl, &wB);
  if (clip) {
    const bool ina = (-1.0f <= Av.x && Av.x <= 1.0f) && (-1.0f <= Av.y && Av.y <= 1.0f) && (-1.0f <= Av.z && Av.z <= 1.0f);
    const bool inb = (-1.0f <= Bv.x && Bv.x <= 1.0f) && (-1.0f <= Bv.y && Bv.y <= 1.0f) && (-1.0f <= Bv.z && Bv.z <= 1.0f);
    if (!ina && !inb) return false;
  }
  const float W = (float)cam.W, H = (float)cam.H;
  const float ax = (Av.x * 0.5f + 0.5f) * W, ay = (Av.y * 0.5f + 0.5f) * H;
  const float bx = (Bv.x * 0.5f + 0.5f) * W, by = (Bv.y * 0.5f + 0.5f) * H;
  s.ws0 = fdiv_rn(1.0f, wA);  // wscale = 1 / (w_A, w_B)   (:83)
  s.ws1 = fdiv_rn(1.0f, wB);
  // draw_line (:50-61): unit step on the major axis, the slope on the other
  const float dx = bx - ax, dy = by - ay;
  const float adx = fabsf(dx), ady = fabsf(dy);
  // along x or along y by selects: the lanes of a wave go both ways
  const bool xm = adx >= ady;
  const float dm = xm ? dx : dy, dn = xm ? dy : dx, km = dm >= 0.0f ? 1.0f : -1.0f, kn = fdiv_rn(km * dn, dm);
  s.kx = xm ? km : kn;
  s.ky = xm ? kn : km;
  s.siz = f2i_sat(xm ? adx : ady);
  int32_t lo, hi;
  wire_major_range(xm ? ax : ay, km, xm ? cam.bias[0] : cam.bias[1], xm ? cam.W : cam.H, s.siz, lo, hi);
  s.ax = ax;
  s.ay = ay;
  s.Az = Av.z;
  s.Bz = Bv.z;
  s.i0 = lo;
  count = hi >= lo ? (uint64_t)((int64_t)hi - lo + 1) : 0;
  return count > 0;
}

// Step i of a wire (:62-64, 84-91): false when its pixel is off the screen.
__device__ __forceinline__ bool wire_step(const Cam& cam, const WSetup& s, long i, int& X, int& Y, int32_t& depth) {
  const float fi = (float)i;
  const float px = s.ax + s.kx * fi, py = s.ay + s.ky * fi;
  const float cor = fi / (float)s.siz;
  X = f2i_sat(floorf(px + cam.bias[0]));
  Y = f2i_sat(floorf(py + cam.bias[1]));
  if (X < 0 || X >= cam.W || Y < 0 || Y >= cam.H) return false;
  float w0 = (1.0f - cor) * s.ws0, w1 = cor * s.ws1;
  const float sum = w0 + w1;
  w0 = w0 / sum;
  w1 = w1 / sum;
  depth = f2i_sat(((w0 * s.Az) + (w1 * s.Bz)) * (float)TINA_MAXDEPTH);
  return true;
}

// Draws the wires of a wave's lanes (count steps of s each) into memory, the steps
// laid end to end, one a lane: of their windows of 64 steps, the part-th of 2^parts_log
// runs.  The first slot whose end is beyond step g owns it: the slots that ended before
// the window, and the ends marked in it below the lane.  mark, slot: LDS of the wave's
// own, 64 words each, mark at -1.
__device__ __forceinline__ void wires_to_memory(const Cam& cam, const WSetup& s, uint64_t count, uint32_t id,
                                                unsigned long long* __restrict__ keys, int* mark, int* slot, int part = 0,
                                                int parts_log = 0) {
  const int lane = __lane_id();
  const unsigned long long live = __ballot(count > 0);
  uint64_t end = count;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t u = __shfl_up(end, d, 64);
    if (lane >= d) end += u;
  }
  const uint64_t total = __shfl(end, 63, 64);
  auto below = [&](unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
  if (count > 0) slot[below(live)] = lane;
  const uint64_t windows = (total + 63) >> 6;
  const uint64_t begin = (windows * (uint64_t)part >> parts_log) << 6, until = (windows * (uint64_t)(part + 1) >> parts_log) << 6;
  int kbase = __popcll(__ballot(count > 0 && end <= begin)), tag = 0;
  for (uint64_t g0 = begin; g0 < until; g0 += 64) {
    // windows are told apart by 31 bits of their number: a mark is read in its own
    tag = (tag + 1) & 0x7fffffff;
    if (count > 0 && end - 1 >= g0 && end - 1 < g0 + 64) mark[(int)(end - 1 - g0)] = tag;
    wave_sync_lds();
    const unsigned long long ends = __ballot(mark[lane] == tag);
    const uint64_t g = g0 + lane;
    const int j = g < total ? slot[kbase + below(ends)] : lane;
    kbase += __popcll(ends);
    WSetup q;
    q.ax = __shfl(s.ax, j);
    q.ay = __shfl(s.ay, j);
    q.kx = __shfl(s.kx, j);
    q.ky = __shfl(s.ky, j);
    q.ws0 = __shfl(s.ws0, j);
    q.ws1 = __shfl(s.ws1, j);
    q.Az = __shfl(s.Az, j);
    q.Bz = __shfl(s.Bz, j);
    q.siz = __shfl(s.siz, j);
    const int64_t i = (int64_t)g + __shfl((int64_t)s.i0 - (int64_t)(end - count), j);
    const uint32_t idj = __shfl(id, j);
    int X, Y;
    int32_t depth;
    if (g < total && wire_step(cam, q, (long)i, X, Y, depth)) {
      const unsigned long long key = pack_key(depth, idj);
      unsigned long long* kp = keys + (long)Y * cam.W + X;
      if (key < __hip_atomic_load(kp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(kp, key);
    }
    wave_sync_lds();
  }
  if (count > 0 || mark[lane] != -1) mark[lane] = -1;
  wave_sync_lds();
}

// Every wire into memory, 64 of them to 2^parts_log waves.
__global__ void __launch_bounds__(kBlock)
k_wires(const float* __restrict__ verts, int n, int parts_log, uint32_t id_base, uint32_t flags, const Cam cam,
        unsigned long long* __restrict__ keys) {
  __shared__ int s_mark[kBlock], s_slot[kBlock];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool clip = (flags & TINA_CLIP) != 0;
  s_mark[threadIdx.x] = -1;
  for (long w = (long)blockIdx.x * (kBlock / 64) + wave; (w >> parts_log) * 64 < n; w += (long)gridDim.x * (kBlock / 64)) {
    WSetup s;
    s.ax = s.ay = s.kx = s.ky = s.ws0 = s.ws1 = s.Az = s.Bz = 0.0f;
    s.siz = s.i0 = 0;
    uint64_t cnt = 0;
    const long f = (w >> parts_log) * 64 + lane;
    if (f < n && !wire_setup(cam, (gf32*)verts, f, clip, s, cnt)) cnt = 0;
    wires_to_memory(cam, s, cnt, id_base + (uint32_t)f, keys, s_mark + 64 * wave, s_slot + 64 * wave,
                    (int)(w & ((1 << parts_log) - 1)), parts_log);
  }
}

// Waves (a power of two, log) that share 64 wires of a call of n: each sets all of them
// up and walks its part of their steps.  Four at least, more while that makes at most
// 64 waves a CU (16 beyond eight): 64 wires a lane of one wave leave a small call with
// a few long-running waves, and one wire a wave (the set-up of 63 lanes idle) made
// 16 k short wires wait for three rounds of waves.  Frames of 1080p, four waves on 64
// wires / one to thirteen wires a wave / so:
//   500 of 600 px 146 / 38 / 33 us, 4 k of 600 157 / 83 / 76, 16 k of 2 px 25 / 30 / 26,
//   16 k of 600 186 / 174 / 167, 60 k of 2 29 / 31 / 28, 200 k of 2 41 / 39 / 39,
//   200 k of 600 816 / 836 / 817, 500 k of 2 62 / 63 / 60 (two waves 64).
inline int wire_parts_log(long n, int ncu) {
  const long chunks = (n + 63) / 64;
  int l = 2;
  while (l < 6 && chunks << (l + 1) <= (l < 3 ? 64L : 16L) * ncu) l++;
  return l;
}

// ---- wires by tile ---------------------------------------------------------------
//
// Each wire's steps land on keys all over the screen, so drawing into memory is
// bound by L2 (a line a step; the 16.6 MB of keys of a 1080p screen do not fit an
// XCD's 4 MB) and by 64-bit atomics (27 G/s).  Calls of many wires therefore go by
// tiles of 32 x 32 pixels whose keys sit in LDS: k_wire_bin lists the wires of
// every tile, k_wire_tile walks each tile's.  What bounds it then is VALU issue in
// the tile pass (about 45 instructions a step, 70 % of its time) and the tiles over
// the middle of the screen, which hold most entries.
// 200 k random wires of 600 px at 1080p: 800 us in memory, 313 by tile (k_wire_bin
// 58, k_wire_tile 255; tiles of 16 pixels some 40 more, of 64 80).  Two workgroups a CU
// take tiles in turn: a workgroup per tile is as fast, but costs 2 us more when all
// groups have drawn their wires.
constexpr int kWireTileLog = 5, kWireTile = 1 << kWireTileLog;

// Calls of this many wires take the two kernels (of twice as many where the keys fit an
// XCD's L2), whose groups go by tile where the call's steps are many (wire_tile_steps).
// Frames of 1080p, drawn by k_wires before / so: 66 k wires of 600, 151, 50, 15 and 5 px
// 409 / 173 us, 196 / 115, 104 / 96, 55 / 57, 37 / 39; 200 k 820 / 318, 373 / 150, 190 /
// 108, 97 / 89, 57 / 60; 500 k 1641 / 655, 694 / 250, 328 / 150, 164 / 110, 92 / 97.  The
// steps are counted on the device, so a call of short wires pays 2 to 5 us for the tile
// pass's empty launch (1.6) and for a raster by k_wire_bin's 16 waves a unit instead of
// 32.  Two ways round that cost more: k_wires first, which puts the long wires by (two
// empty launches, 330 us for the 200 k of 600 px), and workgroups that draw beside those
// that list (long and short in one launch, as slow for short wires).  Below these counts
// short wires are the usual ones (140 k of 2 px at 800 x 450: 25 -> 29).
constexpr int kWireTiledCall = 65536;
constexpr long kXcdL2 = 4L << 20;
inline bool wires_by_tile(long n, long npix) { return n >= (npix * 8 > kXcdL2 ? kWireTiledCall : 2 * kWireTiledCall); }

// Steps of a call from which its wires go by tile; a group of them decides by its share.
// Drawing costs by the step, the tile pass by the tile (a tile with hardly a step takes a
// workgroup some 9 us) and by the wire, which is listed once at least however short.
// The two meet at 2.4 M steps at 1080p, 9 to 10 M at 3840 x 2160 and 1 M at 800 x 450;
// against 3.1 M for any screen and count: 70 k of 50 px at 3840 x 2160 223 -> 138 us, 140 k
// of 31 px 210 -> 156, 200 k of 31 px at 800 x 450 77 -> 55, of 15 px at 1080p 101 -> 89.
inline unsigned long long wire_tile_steps(int ntiles, int n) { return std::max(1100ull * ntiles, 750000ull) + 2ull * n; }

constexpr int kWireSample = 128;  // wires of the sample by which groups decide (k_wire_bin)

// A wire's set-up, one cache line.
struct WireRec {
  float4 a;  // ax, ay, kx, ky
  float4 b;  // ws0, ws1, Az, Bz
  float4 c;  // integers: siz, first and last walked step (none: last < first), then e (below)
  float4 d;  // n0, n1, d0, d1: step i's z is about (n0 + n1 i) / (d0 + d1 i)
};

struct WireJob {
  const float* verts;
  uint64_t* keys;
  uint32_t* chunk_off;
  uint32_t* chunk_cnt;
  uint32_t* entries;
  WireRec* recs;
  uint32_t* gcnt;     // [ngroups] entries of each group
  uint32_t* cursor;   // entries reserved, then the tile pass's next tile; zero between calls
  uint32_t* listed;   // 1: some group has lists; zero between calls
  Cam cam;
  unsigned long long group_steps;  // steps of a group from which it is listed
  int n;
  uint32_t id_base, flags, cap;  // cap: entries there is room for
  int tiles_x, ntiles, ngroups, per;  // per: wires a group
  int sample_stride;  // every so many wires one of the sample
};

// Scratch of wire calls by tile, made for calls of so many wires at a time (room, a power
// of two): as many groups as have a lane for each, and entries for a quarter of the
// screen's tile columns and rows a wire, 24 to 64 (random wires over the whole screen have
// about as many: 22 at 1080p, 44 at 3840 x 2160, where 24 left most of 200 k such wires to
// be drawn, 1,917 us a frame for 628).  1080p: 46 MB for 262,144 wires.  Wires beyond the room are a
// launch pair of their own, which short ones pay for: frames of 500 k of 2 px 83 us with
// a room of 262,144, 70 with one of 524,288 (of 600 px 720, 659; 1 M of 15 px 313, 176).
constexpr int kWireLds = kLdsBudget - 16 * 1024;  // for k_wire_bin's counts by tile (its static LDS is 9 KB)
constexpr int kWireRoom = 1 << 18, kWireMaxRoom = 1 << 20;
constexpr size_t kWireHead = 512;  // bytes at the front that start at zero: the cursor and, on another line, `listed`
struct WireScratch {
  int tiles_x, ntiles, room, entries_a_wire;
  size_t gcnt, chunk_cnt, chunk_off, entries, recs, bytes;  // places in bytes, behind kWireHead
};

// Wires a group of a call of n, n at most the scratch's room: as many groups for every
// unit as give each wire a lane (300 k wires of 5 px: 73 us a frame, 81 where 293 groups
// of 1,024 leave most units with one and some with two), at least 64 wires.
inline int wires_per_group(int n, int ncu) {
  const int k = (n + kBinBlock * ncu - 1) / (kBinBlock * ncu);
  return std::max((n + k * ncu - 1) / (k * ncu), 64);
}

inline WireScratch wire_scratch(int W, int H, int ncu, int n) {
  WireScratch w;
  w.tiles_x = (W + kWireTile - 1) / kWireTile;
  const long ntiles = (long)w.tiles_x * ((H + kWireTile - 1) / kWireTile);
  w.bytes = 0;
  if (4 * ntiles > kWireLds) return w;
  w.ntiles = (int)ntiles;
  long room = kWireRoom;
  while (room < n && room < kWireMaxRoom) room *= 2;
  // the count of all entries has 32 bits: a listed wire has three a tile column or row
  // of its major axis at most (wire_listed)
  w.room = (int)std::min(room, 0xFFFFFFFFL / (4L * (w.tiles_x + ntiles / w.tiles_x + 4)));
  const size_t groups = (size_t)ncu * ((w.room + kBinBlock * ncu - 1) / (kBinBlock * ncu));
  auto place = [&](size_t n) {
    const size_t at = w.bytes;
    w.bytes += (n + 255) & ~(size_t)255;
    return at;
  };
  place(kWireHead);
  w.gcnt = place(4 * groups);
  w.chunk_cnt = place(4 * groups * w.ntiles);
  w.chunk_off = place(4 * groups * w.ntiles);
  w.entries_a_wire = std::min(std::max((w.tiles_x + (int)ntiles / w.tiles_x) / 4, 24), 64);
  w.entries = place(4 * (size_t)w.room * w.entries_a_wire);
  w.recs = place(sizeof(WireRec) * (size_t)w.room);
  return w;
}

inline void wire_scratch_at(const WireScratch& w, void* base, WireJob& j) {
  char* const b = (char*)base;
  j.cursor = (uint32_t*)b;
  j.listed = (uint32_t*)(b + kWireHead / 2);
  j.gcnt = (uint32_t*)(b + w.gcnt);
  j.chunk_cnt = (uint32_t*)(b + w.chunk_cnt);
  j.chunk_off = (uint32_t*)(b + w.chunk_off);
  j.entries = (uint32_t*)(b + w.entries);
  j.recs = (WireRec*)(b + w.recs);
  j.cap = (uint32_t)w.room * (uint32_t)w.entries_a_wire;
  j.tiles_x = w.tiles_x;
  j.ntiles = w.ntiles;
}

// The call's wires [f0, f0 + n), n the scratch's room at most.
inline void wire_job_range(WireJob& j, const float* verts, uint32_t id_base, int f0, int n, int ncu) {
  j.verts = verts + 6 * (size_t)f0;
  j.id_base = id_base + (uint32_t)f0;
  j.n = n;
  j.per = wires_per_group(n, ncu);
  j.ngroups = (n + j.per - 1) / j.per;
  j.sample_stride = std::max(n / kWireSample, 1);
  j.group_steps = wire_tile_steps(j.ntiles, n) * (unsigned long long)j.per / (unsigned long long)n;
}

// Bound on the distance of the binary32 a + k i + bias of a walked step from its
// exact value: three roundings of at most the magnitudes involved (2^-24 each).
__host__ __device__ __forceinline__ double wire_axis_err(float a, float k, int siz, float bias) {
  return 1e-3 + 1e-6 * (fabs((double)a) + fabs((double)k) * (double)siz + fabs((double)bias));
}

// A wire goes by tile while that bound is at most a quarter of a tile (an end some 8
// million pixels away) on both axes: its steps over a tile of the major axis then span
// 48 + 16 pixels of the other, three tiles.  With no such limit a wire that ends 10^9
// pixels away was listed in every tile, and on screens beyond 16 k tiles the entries'
// 32-bit count could wrap.  Such wires are drawn.  False for a NaN.
constexpr double kWireListErr = kWireTile / 4;
__host__ __device__ __forceinline__ bool wire_listed(float ax, float ay, float kx, float ky, int siz, float bx, float by) {
  return wire_axis_err(ax, kx, siz, bx) <= kWireListErr && wire_axis_err(ay, ky, siz, by) <= kWireListErr;
}

// Narrows the steps [lo, hi] to those whose exact position p0 + k i (p0 = a + bias)
// lies within err of [q0, q1].
__host__ __device__ __forceinline__ void wire_clip(double p0, double k, double q0, double q1, double err, double& lo, double& hi) {
  const double l = q0 - err - p0, h = q1 + err - p0;
  if (k == 0.0) {
    if (l > 0.0 || h < 0.0) hi = lo - 1.0;
    return;
  }
  const double ik = 1.0 / k, i0 = l * ik, i1 = h * ik;
  lo = fmax(lo, fmin(i0, i1));
  hi = fmin(hi, fmax(i0, i1));
}

// Every tile a walked step (first to last) of the wire can fall in (and a few beside
// it): along the major axis a tile at a time, the tiles its steps there can reach on
// the other.  w: ax, ay, kx, ky; tx, ty: tiles of the screen.
template <class F>
__host__ __device__ __forceinline__ void wire_tiles(float4 w, int siz, int first, int last, float bx, float by, int tx, int ty,
                                                    F&& visit) {
  const bool xm = fabsf(w.z) == 1.0f;  // unit steps along x
  const double ex = wire_axis_err(w.x, w.z, siz, bx), ey = wire_axis_err(w.y, w.w, siz, by);
  const double px = (double)w.x + (double)bx, py = (double)w.y + (double)by;
  const double pm = xm ? px : py, km = xm ? w.z : w.w, em = xm ? ex : ey;
  const double pn = xm ? py : px, kn = xm ? w.w : w.z, en = xm ? ey : ex;
  const double lo = first, hi = last, tile = kWireTile, inv = 1.0 / kWireTile;
  const int nm = xm ? tx : ty, nn = xm ? ty : tx;
  const double m0 = pm + km * lo, m1 = pm + km * hi;
  const int c0 = (int)fmin(fmax(floor((fmin(m0, m1) - em) * inv), 0.0), (double)nm);
  const int c1 = (int)fmin(fmax(floor((fmax(m0, m1) + em) * inv), -1.0), (double)(nm - 1));
  for (int c = c0; c <= c1; c++) {
    double l = lo, h = hi;
    wire_clip(pm, km, tile * c, tile * (c + 1), em, l, h);
    if (!(l <= h)) continue;
    const double y0 = pn + kn * l, y1 = pn + kn * h;
    const int r0 = (int)fmin(fmax(floor((fmin(y0, y1) - en) * inv), 0.0), (double)nn);
    const int r1 = (int)fmin(fmax(floor((fmax(y0, y1) + en) * inv), -1.0), (double)(nn - 1));
    for (int q = r0; q <= r1; q++) visit(xm ? q * tx + c : c * tx + q);
  }
}

// Group blockIdx.x's wires, at most one a lane (pw to each of the sixteen waves): set
// up, then, where their steps are many, counted per tile and listed per tile (as
// bin_group does for faces); where they are few, drawn into memory, so that the tile
// pass finds nothing to do.  Wires with no length, a value that is not finite or steps
// whose place is not known well enough (wire_listed) have no tiles to find and are
// drawn, as are all of a group whose entries do not fit.
//   Whether their steps are many is decided by a sample of the whole call's wires, the
// same for every group and set up in the lanes that have no wire of their own, as long
// as the group is like it (its steps between 5/8 and 8/5 of the sample's): where groups
// decided each by its own sum, a call near the limit drew some and listed the others and
// paid for both (200 k of 50 px at 3840 x 2160 330 us so, 240 now; drawn 249).
//   MANY: more groups than units; eight waves a SIMD then, two groups a unit (frames of
// 300 k wires of 600 px 456 -> 441 us, 1 M of 2 px 103 -> 98; with fewer groups its two
// spilled registers cost 0.5 us).
template <bool MANY>
__global__ void __launch_bounds__(kBinBlock) __attribute__((amdgpu_waves_per_eu(MANY ? 8 : 4))) k_wire_bin(const WireJob jv) {
  TINA_KERNARG_JOB(WireJob, j, jv);
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t* const cnt = lds;  // [ntiles] counts, then running offsets
  __shared__ unsigned long long s_steps, s_sample;
  __shared__ uint32_t s_base, s_carry, s_wsum[kBinBlock / 64];
  __shared__ int s_mark[kBinBlock], s_slot[kBinBlock];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wbase = tid & ~63, ntiles = j.ntiles;
  constexpr int kWaves = kBinBlock / 64;
  const int pw = (j.per + kWaves - 1) / kWaves;
  const long f0 = (long)blockIdx.x * j.per, f1 = min((long)j.n, f0 + j.per);
  const long f = lane < pw ? f0 + wave * pw + lane : f1;  // this lane's wire
  // or, in kSampleLanes lanes a wave beside them, one of the sample
  constexpr int kSampleLanes = kWireSample / kWaves;
  const bool sampled = pw + kSampleLanes <= 64, samples = sampled && lane >= pw && lane < pw + kSampleLanes;
  const long fs = samples ? min((long)((lane - pw) * kWaves + wave) * j.sample_stride, (long)j.n - 1) : f;
  const bool clip = (j.flags & TINA_CLIP) != 0;
  unsigned long long* const keys = (unsigned long long*)j.keys;
  auto draw = [&](const WSetup& s, uint64_t steps) {
    if (__any(steps > 0)) wires_to_memory(j.cam, s, steps, j.id_base + (uint32_t)f, keys, s_mark + wbase, s_slot + wbase);
  };
  s_mark[tid] = -1;
  if (tid == 0) s_steps = s_sample = 0;
  __syncthreads();
  WSetup s;
  s.ax = s.ay = s.kx = s.ky = s.ws0 = s.ws1 = s.Az = s.Bz = 0.0f;
  s.siz = s.i0 = 0;
  uint64_t steps = 0;
  if ((samples || f < f1) && !wire_setup(j.cam, (gf32*)j.verts, fs, clip, s, steps)) steps = 0;
  // a wave's sums first (a wire counts for 2^24 steps at most, far more than a group's limit)
  const int capped = (int)min(steps, (uint64_t)1 << 24);
  const int wsteps = wave_inclusive_scan(samples ? 0 : capped, lane), wsample = wave_inclusive_scan(samples ? capped : 0, lane);
  if (lane == 63 && wsteps) atomicAdd(&s_steps, (unsigned long long)wsteps);
  if (lane == 63 && wsample) atomicAdd(&s_sample, (unsigned long long)wsample);
  if (samples) steps = 0;
  __syncthreads();
  // uniform: the group's steps and those it would have were it like the sample, times kWireSample
  const unsigned long long own = s_steps * kWireSample, like = s_sample * (unsigned long long)(f1 - f0);
  const unsigned long long decides = sampled && 8 * own > 5 * like && 5 * own < 8 * like ? like : own;
  const bool tiled = decides * j.per >= j.group_steps * kWireSample * (unsigned long long)(f1 - f0);
  if (!tiled) {
    draw(s, steps);
    if (tid == 0) j.gcnt[blockIdx.x] = 0u;  // the tile pass takes no counts from this group
    return;
  }
  for (int t = tid; t < ntiles; t += kBinBlock) cnt[t] = 0;
  __syncthreads();
  const float sum = ((fabsf(s.ax) + fabsf(s.ay)) + (fabsf(s.kx) + fabsf(s.ky))) +
                    ((fabsf(s.ws0) + fabsf(s.ws1)) + (fabsf(s.Az) + fabsf(s.Bz)));
  const bool list = steps > 0 && s.siz > 0 && sum < 1e9f &&
                    wire_listed(s.ax, s.ay, s.kx, s.ky, s.siz, j.cam.bias[0], j.cam.bias[1]);
  const int last = (int)((int64_t)s.i0 + (int64_t)steps - 1);
  auto tiles = [&](auto&& visit) {
    wire_tiles(make_float4(s.ax, s.ay, s.kx, s.ky), s.siz, s.i0, last, j.cam.bias[0], j.cam.bias[1], j.tiles_x, ntiles / j.tiles_x,
               visit);
  };
  if (list) {
    WireRec r;
    r.a = make_float4(s.ax, s.ay, s.kx, s.ky);
    r.b = make_float4(s.ws0, s.ws1, s.Az, s.Bz);
    // z by steps: n / d with n = ws0 Az (1 - c) + ws1 Bz c, d = ws0 (1 - c) + ws1 c, c = i / siz
    const float is = 1.0f / (float)s.siz, n0 = s.ws0 * s.Az, d0 = s.ws0;
    r.d = make_float4(n0, (s.ws1 * s.Bz - n0) * is, d0, (s.ws1 - d0) * is);
    // e: z d computed so, and the reference's own z, are off by less than e (32 roundings
    // of the largest terms); both ends in front of the camera, or no bound
    const float mx = fmaxf(s.ws0, s.ws1), mn = fminf(s.ws0, s.ws1);
    const float e = 32.0f * 5.9604645e-8f * mx * (1.0f + fmaxf(fabsf(s.Az), fabsf(s.Bz))) * (1.0f + mx / mn);
    r.c = make_float4(__int_as_float(s.siz), __int_as_float(s.i0), __int_as_float(last), mn > 0.0f ? e : INFINITY);
    tiles([&](int t) { atomicAdd(&cnt[t], 1u); });
    j.recs[f] = r;
  }
  draw(s, list ? 0 : steps);
  __syncthreads();
  uint32_t* __restrict__ chunk_cnt = j.chunk_cnt + (size_t)blockIdx.x * ntiles;
  uint32_t* __restrict__ chunk_off = j.chunk_off + (size_t)blockIdx.x * ntiles;
  for (int t = tid; t < ntiles; t += kBinBlock) chunk_cnt[t] = cnt[t];
  const uint32_t total = block_exclusive_scan_lds<kBinBlock>(cnt, ntiles, s_wsum, &s_carry);
  if (tid == 0) s_base = atomicAdd(j.cursor, total);  // past the room for some: the sum stays below 2^32
  __syncthreads();
  const uint32_t base = s_base;
  const bool fits = total <= j.cap && base <= j.cap - total;
  if (tid == 0) {
    j.gcnt[blockIdx.x] = fits ? total : 0u;
    if (fits) *j.listed = 1u;
  }
  if (!fits) {
    draw(s, list ? steps : 0);
    return;
  }
  for (int t = tid; t < ntiles; t += kBinBlock) chunk_off[t] = base + cnt[t];
  __syncthreads();
  if (list) tiles([&](int t) { j.entries[base + atomicAdd(&cnt[t], 1u)] = (uint32_t)f; });
}

constexpr int kWireQueue = 128;

// Tile b's wires against its keys in LDS: 64 entries a wave at a time, their steps
// in the tile laid end to end, a step a lane (the lane's wire from a ballot of the
// places where entries end, as in tile_body).  A step whose depth is certainly
// behind the key it would meet is dropped; the others are queued and worked out as
// the reference does in full waves.
template <int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_wire_tile(const WireJob jv) {
  TINA_KERNARG_JOB(WireJob, j, jv);
  if (*j.listed == 0u) return;  // every group has drawn its wires: one word read, 1.6 us
  extern __shared__ uint32_t pre[];  // [ngroups + 1] entries of the tile before each group's
  __shared__ unsigned long long tk[kWireTile * kWireTile];
  __shared__ float4 R0[BLOCK], R1[BLOCK], R2[BLOCK], R3[BLOCK];
  __shared__ int Mark[BLOCK];
  __shared__ uint32_t Q[BLOCK / 64][kWireQueue];  // per wave: up to 127 steps (slot | pixel) and their numbers
  __shared__ int Qi[BLOCK / 64][kWireQueue];
  __shared__ uint32_t s_wsum[BLOCK / 64], s_carry, s_next;
  __shared__ int s_tile;
  const int tid = threadIdx.x, lane = tid & 63, wbase = tid & ~63;
  const int ntiles = j.ntiles, ngroups = j.ngroups;
  const Cam& cam = j.cam;
  const float bx = cam.bias[0], by = cam.bias[1];
  uint32_t* const q = Q[tid >> 6];
  int* const qi = Qi[tid >> 6];
  int tag = 0;  // windows walked: each has a tag of its own
  Mark[tid] = -1;
  for (;;) {
    if (tid == 0) s_tile = (int)atomicAdd(&j.cursor[1], 1u);
    __syncthreads();
    const int t = s_tile;
    if (t >= ntiles) {
      // the last ticket of all: every workgroup has read what the next call starts from
      if (tid == 0 && t == ntiles + (int)gridDim.x - 1) j.cursor[0] = j.cursor[1] = *j.listed = 0u;
      return;
    }
    const int ox = (t % j.tiles_x) << kWireTileLog, oy = (t / j.tiles_x) << kWireTileLog;
    const int tw = min(kWireTile, cam.W - ox), th = min(kWireTile, cam.H - oy);
    const uint32_t total = block_exclusive_scan<BLOCK>(
        ngroups, [&](int c) { return j.gcnt[c] ? j.chunk_cnt[(size_t)c * ntiles + t] : 0u; }, [&](int c, uint32_t o) { pre[c] = o; }, s_wsum,
        &s_carry);
    if (total == 0) continue;
    if (tid == 0) {
      pre[ngroups] = total;
      s_next = 0;
    }
    for (int i = tid; i < kWireTile * kWireTile; i += BLOCK) {
      const int lx = i & (kWireTile - 1), ly = i >> kWireTileLog;
      if (lx < tw && ly < th) tk[i] = j.keys[(size_t)(oy + ly) * cam.W + ox + lx];
    }
    __syncthreads();
    const float fox = (float)ox, foy = (float)oy, ftw = (float)tw, fth = (float)th;
    for (;;) {
      uint32_t b0 = 0;
      if (lane == 0) b0 = atomicAdd(&s_next, 64u);
      b0 = __shfl(b0, 0, 64);
      if (b0 >= total) break;
      const uint32_t v = b0 + lane;
      int cnt = 0;
      WireRec r;
      uint32_t id = 0;
      int s0 = 0;
      if (v < total) {
        int lo = 0, hi = ngroups;  // pre[lo] <= v < pre[hi]
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (pre[mid] <= v) lo = mid; else hi = mid;
        }
        const uint32_t f = j.entries[j.chunk_off[(size_t)lo * ntiles + t] + (v - pre[lo])];
        r = j.recs[f];
        id = j.id_base + f;
        const int siz = __float_as_int(r.c.x);
        double l = __float_as_int(r.c.y), h = __float_as_int(r.c.z);
        wire_clip((double)r.a.x + (double)bx, r.a.z, ox, ox + tw, wire_axis_err(r.a.x, r.a.z, siz, bx), l, h);
        wire_clip((double)r.a.y + (double)by, r.a.w, oy, oy + th, wire_axis_err(r.a.y, r.a.w, siz, by), l, h);
        if (l <= h) {
          s0 = (int)ceil(fmax(l - 0.01, (double)__float_as_int(r.c.y)));
          cnt = ((int)floor(fmin(h + 0.01, (double)__float_as_int(r.c.z))) - s0 + 2) >> 1;  // pairs of steps
        }
      }
      const unsigned long long live = __ballot(cnt > 0);
      const int end = wave_inclusive_scan(cnt > 0 ? cnt : 0, lane);
      const int wtotal = __shfl(end, 63, 64);
      if (cnt > 0) {
        const int slot = wbase + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0u));
        R0[slot] = r.a;
        R1[slot] = r.b;
        R2[slot] = make_float4(r.c.x, __int_as_float(s0 - 2 * (end - cnt)), __uint_as_float(id), r.c.w);
        R3[slot] = r.d;
      }
      wave_sync_lds();
      int qn = 0;     // uniform: pending steps in the queue
      int kbase = 0;  // uniform: entries whose steps all precede the window
      auto exact = [&](int e) {  // queue entry e: its depth as wire_step has it, into the tile
        const uint32_t code = q[e];
        const int k = wbase + (int)(code >> (2 * kWireTileLog));
        const float4 w = R1[k], c = R2[k];
        const float cor = fdiv_rn((float)qi[e], (float)__float_as_int(c.x));
        float w0 = (1.0f - cor) * w.x, w1 = cor * w.y;
        const RcpRN R = rcp_rn(w0 + w1);
        w0 = div_rn(w0, R);
        w1 = div_rn(w1, R);
        const int32_t depth = f2i_sat(((w0 * w.z) + (w1 * w.w)) * (float)TINA_MAXDEPTH);
        atomicMin(&tk[code & (kWireTile * kWireTile - 1)], (unsigned long long)pack_key(depth, __float_as_uint(c.z)));
      };
      for (int g0 = 0; g0 < wtotal; g0 += 64) {
        tag++;
        if (cnt > 0 && end - 1 >= g0 && end - 1 < g0 + 64) Mark[wbase + end - 1 - g0] = tag;
        wave_sync_lds();
        const unsigned long long ends = __ballot(Mark[tid] == tag);
        const int g = g0 + lane;
        bool keep[2] = {false, false};
        uint32_t code[2] = {0u, 0u};
        int i = 0;
        if (g < wtotal) {
          const int k = kbase + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ends >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((uint32_t)ends, 0u));
          const float4 a = R0[wbase + k], c = R2[wbase + k], d = R3[wbase + k];
          i = __float_as_int(c.y) + 2 * g;
          // steps i and i + 1: the latter may lie past the entry's range, where it is
          // a step of the wire all the same (or none, past siz)
  #pragma unroll
          for (int p = 0; p < 2; p++) {
            const float fi = (float)(i + p);
            // the pixel as wire_step has it, less the tile's corner (exact where it matters)
            const float X = floorf((a.x + a.z * fi) + bx) - fox, Y = floorf((a.y + a.w * fi) + by) - foy;
            if ((X >= 0.0f) & (X < ftw) & (Y >= 0.0f) & (Y < fth) & (i + p <= __float_as_int(c.x))) {
              const int at = ((int)Y << kWireTileLog) | (int)X;
              const uint32_t kh = ((const volatile uint32_t*)tk)[2 * at + 1];
              const float kd = (float)(int32_t)(kh ^ 0x80000000u) * 0x1p-30f;
              const float zn = __builtin_fmaf(d.y, fi, d.x), zd = __builtin_fmaf(d.w, fi, d.z);
              keep[p] = !(zn - kd * zd > c.w);
              code[p] = ((uint32_t)k << (2 * kWireTileLog)) | (uint32_t)at;
            }
          }
        }
        kbase += __popcll(ends);
  #pragma unroll
        for (int p = 0; p < 2; p++) {
          const unsigned long long m = __ballot(keep[p]);
          if (keep[p]) {
            const int at = qn + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            q[at] = code[p];
            qi[at] = i + p;
          }
          qn += __popcll(m);
          wave_sync_lds();
          if (qn >= 64) {  // a full wave of them; the rest (at most 63) moves down
            exact(lane);
            const int rest = qn - 64;
            const uint32_t mc = lane < rest ? q[64 + lane] : 0u;
            const int mi = lane < rest ? qi[64 + lane] : 0;
            wave_sync_lds();
            if (lane < rest) {
              q[lane] = mc;
              qi[lane] = mi;
            }
            qn = rest;
            wave_sync_lds();
          }
        }
      }
      if (lane < qn) exact(lane);
      wave_sync_lds();
    }
    __syncthreads();
    for (int i = tid; i < kWireTile * kWireTile; i += BLOCK) {
      const int lx = i & (kWireTile - 1), ly = i >> kWireTileLog;
      if (lx < tw && ly < th) j.keys[(size_t)(oy + ly) * cam.W + ox + lx] = tk[i];
    }
    __syncthreads();
  }
}

// Lanes of a tile's workgroup: 512 while the tiles are several rounds of workgroups
// (256: 414 us against 318 for 200 k wires of 600 px, whose fullest tiles finish
// last), 1,024 on small screens (50 k such wires at 512 x 512: 110 us, 512 lanes 146).
inline int wire_tile_block(int ntiles, int ncu) { return ntiles >= 4 * ncu ? 512 : 1024; }

inline void launch_wire_tile(const WireJob& j, int ncu, hipStream_t s) {
  const int grid = std::min(j.ntiles, 2 * ncu);  // each takes the next tile until none is left
  const size_t lds = (size_t)(j.ngroups + 1) * 4;
  if (wire_tile_block(j.ntiles, ncu) == 512)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_wire_tile<512>), dim3(grid), dim3(512), lds, s, j);
  else
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_wire_tile<1024>), dim3(grid), dim3(1024), lds, s, j);
}

// Pixels won by ids [id_base, id_base + n) take color; with bg_on, empty pixels take bg.
__global__ void __launch_bounds__(kBlock)
k_paint(const uint64_t* __restrict__ keys, long npix, uint32_t id_base, uint32_t n, float cr, float cg, float cb,
        float br, float bgg, float bb, int bg_on, int tonemap, float* __restrict__ img) {
  V3 c = v3(cr, cg, cb), b = v3(br, bgg, bb);
  if (tonemap) {
    c = aces(c);
    b = aces(b);
  }
  for (long P = (long)blockIdx.x * kBlock + threadIdx.x; P < npix; P += (long)gridDim.x * kBlock) {
    const uint64_t k = keys[P];
    if (key_depth(k) >= TINA_MAXDEPTH) {
      if (bg_on) {
        img[3 * P] = b.x;
        img[3 * P + 1] = b.y;
        img[3 * P + 2] = b.z;
      }
    } else if ((uint32_t)k - id_base < n) {
      img[3 * P] = c.x;
      img[3 * P + 1] = c.y;
      img[3 * P + 2] = c.z;
    }
  }
}

}  // namespace tina
