// Launch configurations and the byte layouts of the caller-owned plan,
// workspace and resident-state buffers. Host and device agree on these
// through the structs below (they are passed to kernels by value).
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include <algorithm>

#include "../../include/pgj.h"

namespace pgj {

constexpr int kCap = 4000;   // default PCG iteration cap (exp/asg_gpu_resident_20261103/resident.py:50)

inline size_t align256(size_t v) { return (v + 255) & ~size_t(255); }
inline size_t align8(size_t v) { return (v + 7) & ~size_t(7); }

// ---------------------------------------------------------------- row-march
// The HEX8 row-march kernel maps x to lanes (XPL consecutive x per lane), a
// wavefront marches R element rows over the z-layers of a block, a block has
// W row-waves plus one halo wave and covers W*R node rows and ZC planes.
struct RowMarch {
  int valid;
  int xpl, nl;      // x per lane, active lanes = nx / xpl
  int R, W, ZC;
  int plane;        // 1: plane-carry march (shared in-plane butterflies), 0: node-carry march
  int by, bz;       // blocks along y and z per load
};

// Tuned row-march shapes, keyed by (nz, ny, nx, L, element bytes); set by
// pgj_hex8_set_shape (the autotuner) and consulted by every launch.
// Returns false if unset.
bool tuned_shape(const pgj_grid& g, int L, int es, int* R, int* W, int* ZC, int* plane);

// Radix plan of the compile-time FFT pass `pass` (0 forward xy, 1 z with the Green multiply, 2 inverse xy) of
// the PCG iteration on an n^3 cube in precision es: 0 (not set: the library's choice), 1 (radix 8 first), 2 (z at 64^3
// in registers), 3 (radix 4 first); set by pgj_fft_set_plan (the autotuner) and read at every launch of that pass.
int fft_plan(int n, int es, int pass);

// Row waves and planes per block of the FP64 plane-carry march with two x per lane (246 VGPRs: two waves per SIMD, so a
// CU holds one block of 4 row waves + halo or two of 2 + halo; either way a round of blocks covers 1024 rows). A block
// takes ZC + 1 layers, so the shape with the fewest rounds (ZC + 1) wins; 4 row waves repeat less of the halo, but pay
// only over 16 planes or more and with a last round that is 3/4 full (a CU holds no second block of them). The count of
// CUs is the MI355X's 256. PCG pass, three loads (one load), 4 x 16 / 4 x 32 / 2 x 8 / 2 x 4 row waves x planes: 96^3
// 78 / 74 / 81 / 82 (- / - / 39 / 36) us, 128^3 128 / 150 / 150 / - (44 / - / 50 / -); the node march took 92 (41) and
// 160 (51) at its best shapes, 100 (42) and 161 (58) by its rule. The apply by this rule against the node march by the
// old one, one / three / six loads: 66^3 22 / 48 / 92 against 27 / 58 / 111, 100^3 34 / 92 / 176 against 43 / 111 / 217,
// 128^3 45 / 131 / 248 against 58 / 166 / 329 us.
inline void pair64_shape(int ny, int nz, int L, int* W, int* ZC) {
  int64_t best = -1;
  for (int w : {4, 2, 1}) {
    if (ny % w) continue;
    const int64_t resident = 256 * (8 / (w + 1));
    for (int z = 32; z >= 1; z /= 2) {
      if (nz % z) continue;
      const int64_t blocks = int64_t(ny / w) * (nz / z) * L, rounds = (blocks + resident - 1) / resident;
      if (w == 4 && (z < 16 || 4 * (blocks - (rounds - 1) * resident) < 3 * resident)) continue;
      const int64_t cost = rounds * (z + 1) * (w == 1 ? 4 : 3);  // one row wave per block repeats every row
      if (best < 0 || cost < best) {
        best = cost;
        *W = w;
        *ZC = z;
      }
    }
  }
}

// Shape preferences (R, W, ZC) for L loads per launch. Where no rule below
// sets it, ZC (planes marched by one block) is the largest of 16, 8, 4, 2
// dividing nz that still gives 768 blocks, three per CU: longer marches
// re-read fewer halo planes, but the launch must keep the CUs busy. A tuned
// shape replaces the preferences.
inline RowMarch rowmarch_config(const pgj_grid& g, int L, int es = 8) {
  RowMarch c{};
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  c.xpl = (nx + 63) / 64;
  if (c.xpl > 2 || nx % c.xpl != 0 || ny < 2 || nz < 2 || L < 1) return c;
  c.nl = nx / c.xpl;
  // Default shape (measured on the PCG pass over 32^3..128^3, 1 and 6 loads):
  // the plane-carry march with two row waves (four for FP32 with one x per
  // lane), except FP64 with two x per lane and voxels that are not cubes, whose
  // plane-carry march would spill: that runs the node march.
  const bool pair64 = es == 8 && c.xpl == 2 && g.hx == g.hy && g.hy == g.hz;
  int want_r = 1, want_w = (es == 4 && c.xpl == 1) ? 4 : 2, want_z = 0;
  int want_plane = (es == 4 || c.xpl == 1 || pair64) ? 1 : 0;
  if (pair64) pair64_shape(ny, nz, L, &want_w, &want_z);
  // Launches of few blocks are one block's chain of layers long: one plane per block (two layers instead of three) while
  // every block has a CU of its own, with the fewest row waves that allow it. FP64 stops at two row waves, whose four
  // would only match the two-plane march. PCG pass by this rule against two planes: 16^3 one load 3.8 against 4.9 us,
  // 20^3 4.2 / 4.9, 8^3 six loads 4.2 / 4.9; FP64 apply 16^3 3.4 / 4.3; FP32 apply 16^3 3.1 / 4.2, 32^3 3.6 / 4.3.
  if (c.xpl == 1)
    for (int w = 1; w <= (es == 8 ? 2 : 4); w *= 2)
      if (ny % w == 0 && int64_t(ny / w) * nz * L <= 256) {
        want_w = w;
        want_z = 1;
        break;
      }
  {
    int r = 0, w = 0, z = 0, p = 0;
    if (tuned_shape(g, L, es, &r, &w, &z, &p)) {
      want_r = r; want_w = w; want_z = z; want_plane = p;
    }
  }
  c.plane = want_plane ? 1 : 0;
  // two rows of two x per lane, and two rows of the plane-carry march, exceed 256 VGPRs
  c.R = (want_r == 2 && ny % 2 == 0 && c.xpl == 1 && !c.plane) ? 2 : 1;
  // block = W row-waves + 1 halo wave: at most 5 waves (320 threads, the launch
  // bound of the R = 2, two-x-per-lane and FP64 plane-carry kernels) or 9 waves (576)
  const int wcap = (c.R == 2 || c.xpl == 2 || (c.plane && es == 8)) ? 4 : 8;
  const int wmax = want_w < wcap ? want_w : wcap;
  const int rows = ny / c.R;
  c.W = 1;
  for (int w = wmax; w >= 1; --w)
    if (rows % w == 0) { c.W = w; break; }
  c.by = ny / (c.W * c.R);
  c.ZC = 1;
  if (want_z > 0) {
    for (int z = want_z; z >= 1; --z)
      if (nz % z == 0) { c.ZC = z; break; }
  } else {
    // the longest march (<= 16 planes) that still launches >= 768 blocks (3 per CU), at least 2 planes
    for (int z = 16; z >= 1; z /= 2) {
      if (nz % z != 0) continue;
      c.ZC = z;
      if (int64_t(c.by) * (nz / z) * L >= 768 || z <= 2) break;
    }
  }
  c.bz = nz / c.ZC;
  c.valid = 1;
  return c;
}

inline int hex8_blocks_per_load(const pgj_grid& g, int L, int es = 8) {
  RowMarch c = rowmarch_config(g, L, es);
  if (c.valid) return c.by * c.bz;
  const int64_t n = int64_t(g.nx) * g.ny * g.nz;
  return int((n + 255) / 256);
}

// Upper bound of hex8_blocks_per_load over every shape (W = ZC = R = 1), so
// workspaces stay valid whatever shape is tuned later.
inline int hex8_blocks_bound(const pgj_grid& g) {
  const int64_t n = int64_t(g.nx) * g.ny * g.nz;
  const int64_t rm = int64_t(g.ny) * g.nz;
  const int64_t ref = (n + 255) / 256;
  return int(rm > ref ? rm : ref);
}

// --------------------------------------------------------------------- FFT
// One-dimensional transforms of length n are factored into radices 4, 2, 3, 5, 7.
constexpr int kMaxStages = 12;
struct Factors {
  int n, count;
  int r[kMaxStages];
};

inline Factors factorize(int n) {
  Factors f{};
  f.n = n;
  int m = n;
  while (m % 4 == 0 && f.count < kMaxStages) { f.r[f.count++] = 4; m /= 4; }
  while (m % 2 == 0 && f.count < kMaxStages) { f.r[f.count++] = 2; m /= 2; }
  for (int p : {3, 5, 7})
    while (m % p == 0 && f.count < kMaxStages) { f.r[f.count++] = p; m /= p; }
  if (m != 1) f.count = -1;
  return f;
}

// Radix plan of one axis for the runtime-shaped kernels (fft.hip): the fewest stages of radices 10..2, ties to the plan
// with the largest smallest radix (40 = 8 x 5, 60 = 10 x 6, 75 = 5 x 5 x 3). A group of G lanes carries a line through
// all its stages, so a wavefront holds 64 / G whole lines and a transform needs no block barrier.
constexpr int kMaxAxis = 256;
struct AxisPlan {
  struct Stage {
    int R, nb, Ns, tws;  // radix, butterflies n / R, product of the earlier radices, twiddle step n / (Ns R)
    unsigned mNs;        // j / Ns = j mNs >> 16 for j < n
  } st[4];
  int n, count, G, lpw;  // lanes of a line, lines of a wavefront
  unsigned mG, mL;       // lane / G and lane / lpw as products >> 16
};

inline unsigned magic16(int d) { return 65536u / unsigned(d) + 1; }  // q = x magic >> 16, exact for x d < 65536
inline unsigned magic32(int d) { return unsigned((uint64_t(1) << 32) / unsigned(d) + 1); }  // q = x magic >> 32, d > 1

// Stages of `left` with radices <= cap into r[at...]: the best plan found so far is (best, r).
inline void axis_search(int left, int cap, int at, int lowest, int (&cur)[8], int& best, int& best_low, int (&r)[8]) {
  if (left == 1) {
    if (at < best || (at == best && lowest > best_low)) {
      best = at;
      best_low = lowest;
      for (int i = 0; i < at; ++i) r[i] = cur[i];
    }
    return;
  }
  if (at == 8) return;
  for (int R = cap; R >= 2; --R) {
    if (left % R) continue;
    cur[at] = R;
    axis_search(left / R, R, at + 1, R, cur, best, best_low, r);
  }
}

inline AxisPlan make_axis_plan(int n) {
  AxisPlan a{};
  a.n = n;
  int cur[8], r[8] = {}, best = 9, low = 0;
  axis_search(n, 10, 0, 99, cur, best, low, r);
  a.count = best <= 4 ? best : -1;  // lengths up to 256 take at most three stages
  a.G = 1;
  int Ns = 1;
  for (int s = 0; s < a.count; ++s) {
    a.st[s] = AxisPlan::Stage{r[s], n / r[s], Ns, n / (Ns * r[s]), magic16(Ns)};
    Ns *= r[s];
    if (n / r[s] > a.G) a.G = n / r[s];
  }
  if (a.G > 64) a.G = 64;  // 243 = 9 x 9 x 3 alone: its last stage takes two butterflies per lane
  a.lpw = 64 / a.G;
  a.mG = magic16(a.G);
  a.mL = magic16(a.lpw);
  return a;
}

// Plans of every length up to kMaxAxis, made once (count -1 where a length has another prime factor).
inline const AxisPlan& axis_plan(int n) {
  struct Table {
    AxisPlan p[kMaxAxis + 1];
    Table() {
      for (int i = 1; i <= kMaxAxis; ++i) p[i] = make_axis_plan(i);
    }
  };
  static const Table t;
  static const AxisPlan none{{}, 0, -1, 1, 64, 0, 0};
  return n >= 1 && n <= kMaxAxis ? t.p[n] : none;
}

struct FFTGeom {
  int nz, ny, nx;
  int nkx;          // nx/2 + 1
  int M;            // complex length of the x transform: nx/2 (even nx) or nx (odd)
  int rs;           // row stride of a plane row in LDS (complex): max(nkx, M)
  int64_t nf;       // nz*ny*nkx
  int nkb;          // the workspace holds nkb * ny rows of z pass partials per load
  AxisPlan px, py, pz;
  unsigned mnx, mnkx;  // magic32 of nx and nkx
  int valid;        // some FFT path supports the grid
  int runtime_ok;   // the runtime-shaped kernels (fft.hip) support it
};

// Cubic grids with compile-time-shaped resident FFT kernels (fft_static.hip).
inline bool static_cube(const pgj_grid& g) {
  if (g.nx != g.ny || g.ny != g.nz) return false;
  switch (g.nx) {
    case 16: case 24: case 32: case 48: case 64: case 96: case 128: return true;
    default: return false;
  }
}

constexpr size_t kLdsLimit = 160 * 1024 - 2048;
constexpr int kStageValues = 16;  // complex values a thread holds in one in-place LDS stage

// True when every stage of a batched transform fits the register budget of
// one in-place LDS stage (each thread holds kStageValues/R butterflies).
inline bool stages_fit(const Factors& f, int lines, int threads) {
  for (int s = 0; s < f.count; ++s) {
    const int R = f.r[s];
    if (int64_t(lines) * (f.n / R) > int64_t(threads) * (kStageValues / R)) return false;
  }
  return true;
}

constexpr int kMinChunk = 4;  // frequency columns per block of the runtime z pass: 4, 8 or 16

// Rows of z pass partials per load are partial_chunks(g) ny, at least as many as any z pass of the grid has blocks: the
// compile-time LDS ones N / 2 / kc chunks of N rows and N / kc Nyquist blocks of kc columns or more (kc: the narrowest of
// ZWidths in fft_static.hip), the register-resident ones half as many or fewer of 8 columns, the runtime one at most
// ceil(ny nkx / kMinChunk).
inline int partial_chunks(const pgj_grid& g) {
  int kc = kMinChunk;
  if (static_cube(g)) kc = g.nx == 96 ? 6 : g.nx == 128 ? 8 : 4;
  return (g.nx / 2 + 1 + kc - 1) / kc;
}

inline int64_t half_spectrum(const pgj_grid& g) { return int64_t(g.nz) * g.ny * (g.nx / 2 + 1); }

inline FFTGeom fft_geom(const pgj_grid& g) {
  FFTGeom f{};
  f.nz = g.nz; f.ny = g.ny; f.nx = g.nx;
  f.nkx = g.nx / 2 + 1;
  f.M = (g.nx % 2 == 0) ? g.nx / 2 : g.nx;
  f.rs = f.nkx > f.M ? f.nkx : f.M;
  f.nf = half_spectrum(g);
  const Factors fx = factorize(f.M), fy = factorize(g.ny), fz = factorize(g.nz);
  f.valid = fx.count >= 0 && fy.count >= 0 && fz.count >= 0 && g.nx >= 2 && g.ny >= 2 && g.nz >= 2 &&
            g.nx <= kMaxAxis && g.ny <= kMaxAxis && g.nz <= kMaxAxis;
  const size_t plane = size_t(g.ny) * f.rs * 16;
  const int comps = (3 * plane + 64 <= kLdsLimit) ? 3 : 1;
  if (plane + 64 > kLdsLimit) f.valid = 0;
  const size_t col = size_t(g.nz) * 3 * 16;
  int kc = 1;
  while (kc < f.nkx && size_t(kc + 1) * col + 64 * 8 <= 56 * 1024) ++kc;
  // grids whose planes and columns the block-wide in-place stages of this library once held in registers: the set of
  // supported grids, kept as it was
  if (f.valid)
    f.valid = stages_fit(fx, comps * g.ny, 512) && stages_fit(fy, comps * f.nkx, 512) && stages_fit(fz, 3 * kc, 256);
  f.mnx = magic32(g.nx > 1 ? g.nx : 2);
  f.mnkx = magic32(f.nkx > 1 ? f.nkx : 2);
  f.px = axis_plan(f.M);
  f.py = axis_plan(g.ny);
  f.pz = axis_plan(g.nz);
  f.nkb = partial_chunks(g);
  f.runtime_ok = f.valid;
  if (static_cube(g)) f.valid = 1;
  return f;
}

// Plan buffer: twiddles for x (length M), y, z; then the 6-coefficient symbol.
// rs is the real size: 8 for the FP64 plan, 4 for its FP32 copy.
struct PlanLayout {
  size_t tw_x, tw_y, tw_z, sym, bytes;
};

inline PlanLayout plan_layout(const pgj_grid& g, size_t rs = 8) {
  PlanLayout p{};
  size_t off = 0;
  p.tw_x = off; off = align256(off + size_t(g.nx) * 2 * rs);
  p.tw_y = off; off = align256(off + size_t(g.ny) * 2 * rs);
  p.tw_z = off; off = align256(off + size_t(g.nz) * 2 * rs);
  p.sym = off; off = align256(off + size_t(6) * half_spectrum(g) * rs);
  p.bytes = off;
  return p;
}

// Preconditioner workspace (also the Green part of the resident workspace).
struct PrecondLayout {
  size_t spec;      // L x 3 x nf complex
  size_t pr;        // L x nz x 3 x 2 doubles  (per plane/component: sum r^2, sum r)
  size_t pg;        // L x nkb*ny x 4 doubles  (rz part, sum s_c w_c)
  size_t bytes;
};

inline PrecondLayout precond_layout(const pgj_grid& g, int L, size_t cs = 16) {
  PrecondLayout p{};
  size_t off = 0;
  p.spec = off; off = align256(off + size_t(L) * 3 * half_spectrum(g) * cs);
  p.pr = off; off = align256(off + size_t(L) * g.nz * 6 * 8);
  p.pg = off; off = align256(off + size_t(L) * partial_chunks(g) * g.ny * 4 * 8);
  p.bytes = off;
  return p;
}

// Resident workspace: preconditioner part + operator partials + certify
// partials + per-load refinement scales (cs: complex size of the spectrum).
struct ResidentLayout {
  PrecondLayout pre;
  size_t ppq;       // L x hex8_blocks doubles
  size_t pcert;     // L x nblk x 4 doubles (sum u_c, |r|^2)
  size_t rscale;    // L doubles (FP32 inner solver: |r| of each load's outer residual)
  int nblk_cert;
  size_t bytes;
};

inline ResidentLayout resident_layout(const pgj_grid& g, int L, size_t cs = 16) {
  ResidentLayout r{};
  r.pre = precond_layout(g, L, cs);
  size_t off = r.pre.bytes;
  r.ppq = off; off = align256(off + size_t(L) * hex8_blocks_bound(g) * 8);
  const int64_t n = int64_t(g.nx) * g.ny * g.nz;
  r.nblk_cert = int((n + 255) / 256);
  r.pcert = off; off = align256(off + size_t(L) * r.nblk_cert * 4 * 8);
  r.rscale = off; off = align256(off + size_t(L) * 8);
  r.bytes = off;
  return r;
}

// Loads one resident launch may carry (designs x loads per design).
constexpr int kMaxResidentLoads = 4096;

// Resident state: public blocks first (documented in pgj.h), then private.
struct StateLayout {
  size_t rz, target2, norm, absolute, it, active, bad;
  size_t it_next, active_next, bad_next, first, alpha, stopped, valid, cap, zrows;
  size_t bytes;
};

inline StateLayout state_layout(int L) {
  StateLayout s{};
  size_t off = 0;
  s.rz = off; off += align8(size_t(L) * 8);
  s.target2 = off; off += align8(size_t(L) * 8);
  s.norm = off; off += align8(size_t(L) * 8);
  s.absolute = off; off += align8(size_t(L) * 8);
  s.it = off; off += align8(size_t(L) * 8);
  s.active = off; off += align8(size_t(L));
  s.bad = off; off += align8(size_t(L));
  s.it_next = off; off += align8(size_t(L) * 8);
  s.active_next = off; off += align8(size_t(L));
  s.bad_next = off; off += align8(size_t(L));
  s.first = off; off += align8(size_t(L));
  s.alpha = off; off += align8(size_t(L) * 8);
  s.stopped = off; off += align8(size_t(L));
  s.valid = off; off += align8(size_t(L));
  s.cap = off; off += align8(size_t(L) * 8);
  s.zrows = off; off += align8(size_t(L) * 4);
  s.bytes = align256(off);
  return s;
}

// Device view of the resident state (pointers into one buffer).
struct StateView {
  double* rz;
  double* target2;
  double* norm;
  double* absolute;
  int64_t* it;
  uint8_t* active;
  uint8_t* bad;
  int64_t* it_next;
  uint8_t* active_next;
  uint8_t* bad_next;
  uint8_t* first;
  double* alpha;
  uint8_t* stopped;   // active at the start of this iteration and stopped by its test
  uint8_t* valid;     // this iteration's p.q and r.z were finite and positive (forward pass)
  int64_t* cap;       // iteration cap of the load (set by the set-up)
  int32_t* zrows;     // partial rows the load's last z pass wrote (compile-time cubes)
};

// View of loads [l0, ...) of a state block laid out for L loads.
inline StateView state_view(void* base, int L, int l0 = 0) {
  StateLayout s = state_layout(L);
  char* b = static_cast<char*>(base);
  StateView v;
  v.rz = reinterpret_cast<double*>(b + s.rz) + l0;
  v.target2 = reinterpret_cast<double*>(b + s.target2) + l0;
  v.norm = reinterpret_cast<double*>(b + s.norm) + l0;
  v.absolute = reinterpret_cast<double*>(b + s.absolute) + l0;
  v.it = reinterpret_cast<int64_t*>(b + s.it) + l0;
  v.active = reinterpret_cast<uint8_t*>(b + s.active) + l0;
  v.bad = reinterpret_cast<uint8_t*>(b + s.bad) + l0;
  v.it_next = reinterpret_cast<int64_t*>(b + s.it_next) + l0;
  v.active_next = reinterpret_cast<uint8_t*>(b + s.active_next) + l0;
  v.bad_next = reinterpret_cast<uint8_t*>(b + s.bad_next) + l0;
  v.first = reinterpret_cast<uint8_t*>(b + s.first) + l0;
  v.alpha = reinterpret_cast<double*>(b + s.alpha) + l0;
  v.stopped = reinterpret_cast<uint8_t*>(b + s.stopped) + l0;
  v.valid = reinterpret_cast<uint8_t*>(b + s.valid) + l0;
  v.cap = reinterpret_cast<int64_t*>(b + s.cap) + l0;
  v.zrows = reinterpret_cast<int32_t*>(b + s.zrows) + l0;
  return v;
}

}  // namespace pgj
