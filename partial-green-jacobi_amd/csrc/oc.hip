// Density filters, projections and optimality-criteria (OC) updates.
//
// Two reference variants, both with volume, move and Emin as parameters:
//  - cone: clipped (non-periodic) cone filter, eta-projection, OC with
//    exponent 0.3, lower bound 0.001 and relative-tolerance bisection
//    (exp/asg_sctop_reproduction_20261105/outer.cu:8-39, reproduction.py:69-118);
//  - gaussian: periodic separable Gaussian in scipy's accumulation order,
//    tanh projection, sqrt OC with fixed bisection count
//    (exp/asg_gpu_resident_20261103/outer.cu:7-37, outer.py:26-44).
// Floating-point contraction is disabled so products and sums round like the
// reference's --fmad=false builds and numpy, except where an fma is written out:
// the taps of the fused cone passes, which round once per term instead of twice.
#include <cmath>

#include "layout.h"
#include "pgj_internal.h"

#pragma clang fp contract(off)

namespace pgj {

// bounds layout (cone):     [lo, hi, running (1/0), bisection count]
// bounds layout (gaussian): [lo, hi]

__global__ __launch_bounds__(256) void cone_filter_kernel(const double* x, const int* off, const double* w, int m, int n,
                                                          double* y, const double* bounds, int conditional) {
  const int64_t N = int64_t(n) * n * n;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N || (conditional && bounds[2] == 0.0)) return;
  const int xx = int(i % n), yy = int((i / n) % n), zz = int(i / (int64_t(n) * n));
  double sum = 0.0;
  for (int j = 0; j < m; ++j) {
    const int xj = xx + off[3 * j], yj = yy + off[3 * j + 1], zj = zz + off[3 * j + 2];
    if (xj >= 0 && xj < n && yj >= 0 && yj < n && zj >= 0 && zj < n) sum += w[j] * x[(int64_t(zj) * n + yj) * n + xj];
  }
  y[i] = sum;
}

// eta-projection: rho = (tanh(b eta) + tanh(b (t/hs - eta))) / den, with volume partials.
__global__ __launch_bounds__(256) void cone_project_kernel(const double* t, const double* hs, double* ph, double* dp,
                                                           double* a, const double* bounds, int64_t N, double beta,
                                                           double eta, double emin, int conditional, double* vpart) {
  __shared__ double red[8];
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (conditional && bounds[2] == 0.0) return;
  double rho = 0.0;
  if (i < N) {
    const double den = tanh(beta * eta) + tanh(beta * (1 - eta));
    const double q = tanh(beta * (t[i] / hs[i] - eta));
    rho = (tanh(beta * eta) + q) / den;
    ph[i] = rho;
    dp[i] = beta * (1 - q * q) / den;
    a[i] = emin + (1 - emin) * rho * rho * rho;
  }
  if (vpart) {
    const double s = block_sum(rho, red);
    if (threadIdx.x == 0) vpart[blockIdx.x] = s;
  }
}

// g_in = dp (3 (1-Emin) ph^2) e / hs ; dv_in = dp / hs
__global__ __launch_bounds__(256) void cone_prepare_kernel(const double* dp, const double* ph, const double* e,
                                                           const double* hs, double emin, int64_t N, double* gin,
                                                           double* dvin) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double c = 3 * (1 - emin) * (ph[i] * ph[i]);
  gin[i] = dp[i] * c * e[i] / hs[i];
  dvin[i] = dp[i] / hs[i];
}

// g /= n^3 ; ratio = -g / dv ; reset bounds for the bisection.
__global__ __launch_bounds__(256) void cone_ratio_kernel(double* g, const double* dv, int64_t N, double* ratio,
                                                         double* bounds) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i == 0) {
    bounds[0] = 0.0;
    bounds[1] = 1e9;
    bounds[2] = 1.0;
    bounds[3] = 0.0;
  }
  if (i >= N) return;
  const double gv = g[i] / double(N);
  g[i] = gv;
  ratio[i] = -gv / dv[i];
}

__global__ __launch_bounds__(256) void cone_candidate_kernel(const double* x, const double* ratio, const double* bounds,
                                                             double move, double* y, int64_t N) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N || bounds[2] == 0.0) return;
  const double mid = 0.5 * (bounds[0] + bounds[1]);
  const double v = x[i] * pow(fmax(1e-10, ratio[i] / mid), 0.3);
  y[i] = fmax(0.001, fmax(x[i] - move, fmin(1.0, fmin(x[i] + move, v))));
}

__global__ void cone_bisect_kernel(const double* vpart, int nblk, int64_t N, double* b, double target) {
  if (b[2] == 0.0) return;
  const double s = wave_reduce_partials(vpart, nblk, 1);
  if (threadIdx.x == 0) {
    const double volume = s / double(N);
    const double mid = 0.5 * (b[0] + b[1]);
    if (volume > target) b[0] = mid;
    else b[1] = mid;
    b[3] += 1.0;
    b[2] = ((b[1] - b[0]) / (b[1] + b[0]) > 1e-4 && b[1] > 1e-40) ? 1.0 : 0.0;
  }
}

// ------------------------------------------------- fused cone filter passes
// The cone filter is a short stencil (93 taps at rmin 3) whose 93 global loads per node, not their sums, took the
// time (30 us of a 47 us bisection round at 64^3: 0.8 TB/s of cache reads and a bounds test per tap). The fused
// passes stage a 16 x 8 x 8 tile and its halo in LDS once, zero outside the cube, and take the taps from there in
// the stencil's order, so every sum has the terms and order of cone_filter_kernel (a skipped tap adds +0; each term
// is one FMA, rounded once instead of twice). What is left is bound by FP64 issue.
// They exist for a reach of at most kConeReach planes (34 KiB of LDS there).
constexpr int kConeReach = 3;
constexpr int kTX = 16, kTY = 8, kTZ = 8, kConeThreads = 512, kPer = kTX * kTY * kTZ / kConeThreads;

struct ConeStencil {
  int n, m;
  const int* off;       // (m, 3) dx, dy, dz
  const double* w;
};

// eta-projection: rho = (te + tanh(beta (t/hs - eta))) / den with te = tanh(beta eta), den = te + tanh(beta (1 - eta)).
struct ConeProjection {
  double beta, eta, te, den;
};

template <int R>
struct ConeTile {
  static constexpr int SX = kTX + 2 * R, SY = kTY + 2 * R, SZ = kTZ + 2 * R, SIZE = SX * SY * SZ;
  static constexpr int PER = (SIZE + kConeThreads - 1) / kConeThreads;
  // Stages make(fetch(node), node, own) of the tile and its halo; own: the node is one of the tile's. Every fetch of a
  // thread is issued (from a clamped, in-bounds node) before the first make, so their latencies overlap.
  template <typename Fetch, typename Make>
  __device__ static void stage(double* t, int n, int x0, int y0, int z0, Fetch fetch, Make make) {
    decltype(fetch(int64_t(0))) raw[PER];
    auto coords = [&](int k, int& x, int& y, int& z, bool& own) {
      const int e = min(int(threadIdx.x) + k * kConeThreads, SIZE - 1);
      const int ex = e % SX, ey = (e / SX) % SY, ez = e / (SX * SY);
      x = x0 + ex - R; y = y0 + ey - R; z = z0 + ez - R;
      own = ex >= R && ex < R + kTX && ey >= R && ey < R + kTY && ez >= R && ez < R + kTZ;
    };
    int x, y, z;
    bool own;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      coords(k, x, y, z, own);
      const int cx = min(max(x, 0), n - 1), cy = min(max(y, 0), n - 1), cz = min(max(z, 0), n - 1);
      raw[k] = fetch((int64_t(cz) * n + cy) * n + cx);
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = int(threadIdx.x) + k * kConeThreads;
      if (e >= SIZE) break;
      coords(k, x, y, z, own);
      double v = 0.0;
      if (x >= 0 && x < n && y >= 0 && y < n && z >= 0 && z < n) v = make(raw[k], (int64_t(z) * n + y) * n + x, own);
      t[e] = v;
    }
  }
  // sums[k] of node (x, y, z + k) of the tile, k < kPer. The taps are uniform: eight of them are fetched through the
  // scalar cache at a time and their values read from LDS before the first is used (one at a time, every tap waited
  // for both: 64^3, 18.9 us a pass).
  template <int COUNT>
  __device__ static __forceinline__ void taps(const double* p, const int* __restrict__ off, const double* __restrict__ w,
                                              double (&sums)[kPer]) {
    double v[COUNT][kPer];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) {
      const double* q = p + (off[3 * u + 2] * SY + off[3 * u + 1]) * SX + off[3 * u];
#pragma unroll
      for (int k = 0; k < kPer; ++k) v[u][k] = q[k * SY * SX];
    }
#pragma unroll
    for (int u = 0; u < COUNT; ++u)
#pragma unroll
      for (int k = 0; k < kPer; ++k) sums[k] = fma(w[u], v[u][k], sums[k]);
  }
  __device__ static void filter(const double* t, const ConeStencil& c, int lx, int ly, int lz, double (&sums)[kPer]) {
    const double* p = t + ((lz + R) * SY + ly + R) * SX + lx + R;
#pragma unroll
    for (int k = 0; k < kPer; ++k) sums[k] = 0.0;
    int j = 0;
    for (; j + 8 <= c.m; j += 8) taps<8>(p, c.off + 3 * j, c.w + j, sums);
    if (c.m & 4) {
      taps<4>(p, c.off + 3 * j, c.w + j, sums);
      j += 4;
    }
    for (; j < c.m; ++j) taps<1>(p, c.off + 3 * j, c.w + j, sums);
  }
};

// This thread's nodes: (lx, ly, lz + k) of the tile, k < kPer.
__device__ __forceinline__ void cone_local(int& lx, int& ly, int& lz) {
  lx = threadIdx.x % kTX;
  ly = (threadIdx.x / kTX) % kTY;
  lz = threadIdx.x / (kTX * kTY) * kPer;
}

// t = filter(x) and its projection.
template <int R>
__global__ __launch_bounds__(kConeThreads) void cone_physical_kernel(ConeStencil c, const double* x, const double* hs,
                                                                     ConeProjection pr, double emin, double* t,
                                                                     double* ph, double* dp, double* a) {
  __shared__ double tile[ConeTile<R>::SIZE];
  const int n = c.n, x0 = blockIdx.x * kTX, y0 = blockIdx.y * kTY, z0 = blockIdx.z * kTZ;
  ConeTile<R>::stage(
      tile, n, x0, y0, z0, [&](int64_t i) { return x[i]; }, [](double v, int64_t, bool) { return v; });
  __syncthreads();
  int lx, ly, lz;
  cone_local(lx, ly, lz);
  double f[kPer];
  ConeTile<R>::filter(tile, c, lx, ly, lz, f);
  if (x0 + lx >= n || y0 + ly >= n) return;
  for (int k = 0; k < kPer && z0 + lz + k < n; ++k) {
    const int64_t i = (int64_t(z0 + lz + k) * n + y0 + ly) * n + x0 + lx;
    const double q = tanh(pr.beta * (f[k] / hs[i] - pr.eta));
    const double rho = (pr.te + q) / pr.den;
    t[i] = f[k];
    ph[i] = rho;
    dp[i] = pr.beta * (1 - q * q) / pr.den;
    a[i] = emin + (1 - emin) * rho * rho * rho;
  }
}

// Unevaluated sums of two doubles (the second below half an ulp of the first), products by FMA.
struct Two {
  double hi, lo;
};
__device__ __forceinline__ Two two_mul(Two a, Two b) {
  const double p = a.hi * b.hi;
  const double e = fma(a.hi, b.hi, -p) + (a.hi * b.lo + a.lo * b.hi);
  const double h = p + e;
  return {h, e - (h - p)};
}

// q^0.3 (q > 0, or q^-0.3 with INV) as a sum of two doubles: the power, then one Newton step on p^10 = q^3 in two
// doubles. A correction that is not finite (a power of 0 or infinity, p^10 out of range) is left out.
template <bool INV>
__device__ __forceinline__ Two root03(double q) {
  const double p = pow(q, INV ? -0.3 : 0.3);
  const Two b{p, 0.0}, b2 = two_mul(b, b), b4 = two_mul(b2, b2), b10 = two_mul(two_mul(b4, b4), b2);
  const Two c{q, 0.0}, c3 = two_mul(two_mul(c, c), c);
  double e;
  if (INV) {
    const Two u = two_mul(b10, c3);
    e = p * ((1.0 - u.hi) - u.lo) / 10.0;
  } else {
    e = p * (((c3.hi - b10.hi) + (c3.lo - b10.lo)) / b10.hi) / 10.0;
  }
  return {p, isfinite(e) && fabs(e) <= 1e-12 * p ? e : 0.0};
}

// g = filter(dp 3 (1 - Emin) ph^2 e / hs) / n^3, dv = filter(dp / hs), ratio = -g / dv; bounds reset. root: ratio^0.3
// (0 where ratio is not positive) as (hi, lo) pairs for cone_round_kernel.
template <int R>
__global__ __launch_bounds__(kConeThreads) void cone_gradient_kernel(ConeStencil c, const double* dp, const double* ph,
                                                            const double* e, const double* hs, double emin, double* g,
                                                            double* dv, double* ratio, double2* root, double* bounds) {
  __shared__ double tile[ConeTile<R>::SIZE];
  const int n = c.n, x0 = blockIdx.x * kTX, y0 = blockIdx.y * kTY, z0 = blockIdx.z * kTZ;
  if (threadIdx.x == 0 && blockIdx.x + blockIdx.y + blockIdx.z == 0) {
    bounds[0] = 0.0;
    bounds[1] = 1e9;
    bounds[2] = 1.0;
    bounds[3] = 0.0;
  }
  int lx, ly, lz;
  cone_local(lx, ly, lz);
  double fg[kPer], fv[kPer];
  struct Raw {
    double dp, ph, e, hs;
  };
  ConeTile<R>::stage(
      tile, n, x0, y0, z0, [&](int64_t i) { return Raw{dp[i], ph[i], e[i], hs[i]}; },
      [&](const Raw& v, int64_t, bool) {
        const double cf = 3 * (1 - emin) * (v.ph * v.ph);
        return v.dp * cf * v.e / v.hs;
      });
  __syncthreads();
  ConeTile<R>::filter(tile, c, lx, ly, lz, fg);
  __syncthreads();
  ConeTile<R>::stage(
      tile, n, x0, y0, z0, [&](int64_t i) { return double2{dp[i], hs[i]}; },
      [](const double2& v, int64_t, bool) { return v.x / v.y; });
  __syncthreads();
  ConeTile<R>::filter(tile, c, lx, ly, lz, fv);
  if (x0 + lx >= n || y0 + ly >= n) return;
  const double N = double(int64_t(n) * n * n);
  for (int k = 0; k < kPer && z0 + lz + k < n; ++k) {
    const int64_t i = (int64_t(z0 + lz + k) * n + y0 + ly) * n + x0 + lx;
    const double gv = fg[k] / N;
    g[i] = gv;
    dv[i] = fv[k];
    const double q = -gv / fv[k];
    ratio[i] = q;
    const Two p = q > 0.0 ? root03<false>(q) : Two{0.0, 0.0};
    root[i] = double2{p.hi, p.lo};
  }
}

// One bisection step on bounds values b from the volume sum s of its candidate.
__device__ __forceinline__ void cone_bisect_step(double (&b)[4], double s, double N, double target) {
  const double volume = s / N;
  const double mid = 0.5 * (b[0] + b[1]);
  if (volume > target) b[0] = mid;
  else b[1] = mid;
  b[3] += 1.0;
  b[2] = ((b[1] - b[0]) / (b[1] + b[0]) > 1e-4 && b[1] > 1e-40) ? 1.0 : 0.0;
}

// One round of the bisection in one launch: every block finishes the previous round's bisection for itself from the
// volume partials vprev (none in the first round), block 0 leaves the bounds for the next round in `out` (not the
// buffer the others read), then candidate, filter, projection and the volume partials of this round. The candidate
// x max(1e-10, ratio / mid)^0.3 = x max(floor, ratio^0.3 mid^-0.3) is evaluated on the halo too, from the two
// factors kept to two doubles each: a few FMAs per node and no larger an error than the power of the rounded quotient
// (a power per node and round, 2.8 with the halo, was 7 us of the launch). 64^3, rmin 3: 47 us in four launches
// before, 11 us now.
template <int R>
__global__ __launch_bounds__(kConeThreads) void cone_round_kernel(ConeStencil c, const double* x, const double2* root,
                                                                  const double* hs, ConeProjection pr, double floor03,
                                                                  double move, double target, const double* in,
                                                                  const double* vprev, double* out, double* vpart,
                                                                  double* y) {
  __shared__ double tile[ConeTile<R>::SIZE];
  __shared__ double red[kConeThreads / 64], sb[3];
  const int n = c.n, x0 = blockIdx.x * kTX, y0 = blockIdx.y * kTY, z0 = blockIdx.z * kTZ;
  const int nblk = gridDim.x * gridDim.y * gridDim.z, blk = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  if (threadIdx.x < 64) {
    double b[4] = {in[0], in[1], in[2], in[3]};
    if (vprev && b[2] != 0.0)
      cone_bisect_step(b, wave_reduce_partials(vprev, nblk, 1), double(int64_t(n) * n * n), target);
    const Two f = root03<true>(0.5 * (b[0] + b[1]));
    if (threadIdx.x == 0) {
      sb[0] = f.hi;
      sb[1] = f.lo;
      sb[2] = b[2];
      if (blk == 0)
        for (int k = 0; k < 4; ++k) out[k] = b[k];
    }
  }
  __syncthreads();
  if (sb[2] == 0.0) return;
  const double mh = sb[0], ml = sb[1];
  struct Raw {
    double x;
    double2 p;
  };
  ConeTile<R>::stage(
      tile, n, x0, y0, z0, [&](int64_t i) { return Raw{x[i], root[i]}; },
      [&](const Raw& r, int64_t i, bool own) {
        const double e = r.p.x * ml + r.p.y * mh;
        const double v = r.x * fmax(floor03, fma(r.p.x, mh, isfinite(e) ? e : 0.0));
        const double yi = fmax(0.001, fmax(r.x - move, fmin(1.0, fmin(r.x + move, v))));
        if (own) y[i] = yi;
        return yi;
      });
  __syncthreads();
  int lx, ly, lz;
  cone_local(lx, ly, lz);
  double f[kPer];
  ConeTile<R>::filter(tile, c, lx, ly, lz, f);
  double rho = 0.0;
  if (x0 + lx < n && y0 + ly < n)
    for (int k = 0; k < kPer && z0 + lz + k < n; ++k) {
      const int64_t i = (int64_t(z0 + lz + k) * n + y0 + ly) * n + x0 + lx;
      const double q = tanh(pr.beta * (f[k] / hs[i] - pr.eta));
      rho += (pr.te + q) / pr.den;
    }
  const double s = block_sum(rho, red);
  if (threadIdx.x == 0) vpart[blk] = s;
}

// The bisection of the last round of a sequence, into the caller's bounds.
__global__ void cone_rounds_finish(const double* in, const double* vpart, int nblk, int64_t N, double target,
                                   double* bounds) {
  double b[4] = {in[0], in[1], in[2], in[3]};
  if (b[2] != 0.0) cone_bisect_step(b, wave_reduce_partials(vpart, nblk, 1), double(N), target);
  if (threadIdx.x == 0)
    for (int k = 0; k < 4; ++k) bounds[k] = b[k];
}

// max |a - b| partials and finish (order independent)
__global__ __launch_bounds__(256) void absmax_partials(const double* a, const double* b, int64_t N, double* part) {
  __shared__ double red[8];
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double v = i < N ? fabs(a[i] - b[i]) : 0.0;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) m = fmax(m, red[k]);
    part[blockIdx.x] = m;
  }
}

__global__ void absmax_finish(const double* part, int nblk, double* out) {
  double v = 0.0;
  for (int k = threadIdx.x; k < nblk; k += 64) v = fmax(v, part[k]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  if (threadIdx.x == 0) out[0] = v;
}

// ------------------------------------------------------------------ gaussian
// Periodic correlation along one axis in scipy's symmetric order:
// y = w[r] x[i] + sum_{k=r..1} (x[i-k] + x[i+k]) w[r+k].
__global__ __launch_bounds__(256) void gauss_axis_kernel(const double* x, const double* w, int radius, int n, int axis,
                                                         double* y) {
  const int64_t N = int64_t(n) * n * n;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int64_t stride = axis == 0 ? int64_t(n) * n : (axis == 1 ? n : 1);
  const int coord = int((i / stride) % n);
  double v = x[i] * w[radius];
  for (int k = radius; k >= 1; --k) {
    int lo = (coord - k) % n;
    if (lo < 0) lo += n;
    const int hi = (coord + k) % n;
    v += (x[i + int64_t(lo - coord) * stride] + x[i + int64_t(hi - coord) * stride]) * w[radius + k];
  }
  y[i] = v;
}

__global__ __launch_bounds__(256) void gauss_project_kernel(const double* t, double beta, double* ph, double* dp,
                                                            double* a, int64_t N, double emin, double* vpart) {
  __shared__ double red[8];
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double p = 0.0;
  if (i < N) {
    const double den = 2 * tanh(beta / 2);
    const double q = tanh(beta * (t[i] - 0.5));
    p = (tanh(beta / 2) + q) / den;
    ph[i] = p;
    dp[i] = beta * (1 - q * q) / den;
    a[i] = emin + (1 - emin) * (p * p * p);
  }
  if (vpart) {
    const double s = block_sum(p, red);
    if (threadIdx.x == 0) vpart[blockIdx.x] = s;
  }
}

// g_in = dp p (1-Emin) ph^2 e  (left-to-right as the reference)
__global__ __launch_bounds__(256) void gauss_prepare_kernel(const double* dp, const double* ph, const double* e,
                                                            double emin, double penal, int64_t N, double* gin) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  gin[i] = dp[i] * penal * (1 - emin) * (ph[i] * ph[i]) * e[i];
}

// ratio = max(g,1e-30)/max(dv,1e-30), block maxima of ratio
__global__ __launch_bounds__(256) void gauss_ratio_kernel(const double* g, const double* dv, int64_t N, double* ratio,
                                                          double* part) {
  __shared__ double red[8];
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double v = 0.0;
  if (i < N) {
    v = fmax(g[i], 1e-30) / fmax(dv[i], 1e-30);
    ratio[i] = v;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) m = fmax(m, red[k]);
    part[blockIdx.x] = m;
  }
}

__global__ void gauss_bounds_kernel(const double* part, int nblk, double* bounds) {
  double v = 0.0;
  for (int k = threadIdx.x; k < nblk; k += 64) v = fmax(v, part[k]);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  if (threadIdx.x == 0) {
    bounds[0] = 0.0;
    bounds[1] = v * 1e4;
  }
}

__global__ __launch_bounds__(256) void gauss_candidate_kernel(const double* x, const double* ratio, const double* bounds,
                                                              double move, double* y, int64_t N) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double lam = fmax((bounds[0] + bounds[1]) * 0.5, 1e-30);
  const double lo = fmax(0.0, x[i] - move), hi = fmin(1.0, x[i] + move);
  y[i] = fmin(hi, fmax(lo, x[i] * sqrt(ratio[i] / lam)));
}

__global__ void gauss_bisect_kernel(const double* vpart, int nblk, int64_t N, double* b, double target) {
  const double s = wave_reduce_partials(vpart, nblk, 1);
  if (threadIdx.x == 0) {
    const double mid = (b[0] + b[1]) * 0.5;
    if (s / double(N) > target) b[0] = mid;
    else b[1] = mid;
  }
}

// ------------------------------------------------------- gaussian in two passes
// The three axis passes as two launches: z on columns staged in LDS, then y and x on strips of a z-plane staged in
// LDS with their y halo. Each line is summed in gauss_axis_kernel's order. A bisection round (candidate, three axis
// passes, projection, bisection: six launches, bound by their issue from the host at 38 us a round) is two.
constexpr int kGaussCols = 16;
// Rows of a strip: 8 up to n = 48, where 16 leave a launch with half a block per CU or less. The update with 8 and 16 rows
// (us): 24^3 399 / 443, 32^3 432 / 472, 40^3 564 / 627, 48^3 666 / 650; above the line 56^3 779 / 837, 64^3 795 / 914,
// 96^3 1932 / 2108, so the line could lie higher.
__host__ __device__ inline int gauss_rows(int n) { return n <= 48 ? 8 : 16; }

// Weighted symmetric sum at `i` of a periodic line of n values with stride `st` in LDS (radius <= n).
__device__ __forceinline__ double gauss_line(const double* line, int st, int i, int n, const double* w, int radius) {
  double v = line[i * st] * w[radius];
  for (int k = radius; k >= 1; --k) {
    const int lo = i - k < 0 ? i - k + n : i - k, hi = i + k >= n ? i + k - n : i + k;
    v += (line[lo * st] + line[hi * st]) * w[radius + k];
  }
  return v;
}

// One bisection step on (lo, hi).
__device__ __forceinline__ void gauss_bisect_step(double (&b)[2], double s, double N, double target) {
  const double mid = (b[0] + b[1]) * 0.5;
  if (s / N > target) b[0] = mid;
  else b[1] = mid;
}

// z pass. CAND: the input is the OC candidate of x at this round's multiplier, whose bounds every block finishes from
// the previous round's volume partials (none in the first round); block 0 leaves them in `out`.
template <bool CAND>
__global__ __launch_bounds__(256) void gauss_z_kernel(const double* x, const double* ratio, double move, double target,
                                                      const double* in, const double* vprev, int nblk, double* out,
                                                      const double* w, int radius, int n, double* y, double* z) {
  extern __shared__ double col[];
  __shared__ double slam;
  const int64_t NN = int64_t(n) * n;
  if (CAND) {
    if (threadIdx.x < 64) {
      double b[2] = {in[0], in[1]};
      if (vprev) gauss_bisect_step(b, wave_reduce_partials(vprev, nblk, 1), double(NN * n), target);
      if (threadIdx.x == 0) {
        slam = fmax((b[0] + b[1]) * 0.5, 1e-30);
        if (blockIdx.x == 0) {
          out[0] = b[0];
          out[1] = b[1];
        }
      }
    }
    __syncthreads();
  }
  const int c = threadIdx.x % kGaussCols;
  const int64_t p = int64_t(blockIdx.x) * kGaussCols + c;
  const bool on = p < NN;
  for (int k = threadIdx.x / kGaussCols; k < n; k += 256 / kGaussCols) {
    double v = 0.0;
    if (on) {
      const int64_t i = k * NN + p;
      v = x[i];
      if (CAND) {
        const double lo = fmax(0.0, v - move), hi = fmin(1.0, v + move);
        v = fmin(hi, fmax(lo, v * sqrt(ratio[i] / slam)));
        y[i] = v;
      }
    }
    col[k * kGaussCols + c] = v;
  }
  __syncthreads();
  if (!on) return;
  for (int k = threadIdx.x / kGaussCols; k < n; k += 256 / kGaussCols)
    z[k * NN + p] = gauss_line(col + c, kGaussCols, k, n, w, radius);
}

// y and x passes of gauss_rows(n) rows of a z-plane (inv: 2^32 / n rounded up, for the division by n). VOLUME: the
// projected density's sum per block instead of the field.
template <bool VOLUME>
__global__ __launch_bounds__(256) void gauss_yx_kernel(const double* z, const double* w, int radius, int n,
                                                       unsigned inv, double beta, double* y, double* vpart) {
  extern __shared__ double strip[];
  __shared__ double red[4];
  const int full = gauss_rows(n), y0 = blockIdx.x * full, rows = min(full, n - y0);
  double* mid = strip + (full + 2 * radius) * n;
  const double* plane = z + int64_t(blockIdx.y) * n * n;
  const int tall = rows + 2 * radius;
  for (int e = threadIdx.x; e < tall * n; e += 256) {
    const int q = __umulhi(e, inv);   // e / n
    int r = y0 - radius + q;
    r = r < 0 ? r + n : r;
    r = r >= n ? r - n : r;
    strip[e] = plane[int64_t(r) * n + (e - q * n)];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < rows * n; e += 256) {
    const double* p = strip + e + radius * n;   // row e / n of the strip's own rows
    double v = p[0] * w[radius];
    for (int k = radius; k >= 1; --k) v += (p[-k * n] + p[k * n]) * w[radius + k];
    mid[e] = v;
  }
  __syncthreads();
  double sum = 0.0;
  const double den = 2 * tanh(beta / 2), tb = tanh(beta / 2);
  for (int e = threadIdx.x; e < rows * n; e += 256) {
    const int row = __umulhi(e, inv) * n;
    const double v = gauss_line(mid + row, 1, e - row, n, w, radius);
    if (VOLUME) sum += (tb + tanh(beta * (v - 0.5))) / den;
    else y[(int64_t(blockIdx.y) * n + y0) * n + e] = v;
  }
  if (VOLUME) {
    const double t = block_sum(sum, red);
    if (threadIdx.x == 0) vpart[blockIdx.y * gridDim.x + blockIdx.x] = t;
  }
}

__global__ void gauss_rounds_finish(const double* in, const double* vpart, int nblk, int64_t N, double target,
                                    double* bounds) {
  double b[2] = {in[0], in[1]};
  gauss_bisect_step(b, wave_reduce_partials(vpart, nblk, 1), double(N), target);
  if (threadIdx.x == 0) {
    bounds[0] = b[0];
    bounds[1] = b[1];
  }
}

}  // namespace pgj

using namespace pgj;

namespace {
int blocks_of(int64_t N) { return int((N + 255) / 256); }

// LDS of the strips of gauss_yx_kernel; the fused passes run where it and the columns fit 64 KiB.
size_t gauss_lds(int n, int radius) { return (2 * size_t(gauss_rows(n)) + 2 * radius) * n * 8; }
bool gauss_fused(int n, int radius) {
  return radius <= n && gauss_lds(n, radius) <= 65536 - 64 && size_t(n) * kGaussCols * 8 <= 65536 - 64;
}
int gauss_strips(int n) { return (n + gauss_rows(n) - 1) / gauss_rows(n); }
unsigned gauss_inv(int n) { return unsigned((0xffffffffull + n) / n); }
int gauss_columns(int n) { return int((int64_t(n) * n + kGaussCols - 1) / kGaussCols); }
}

extern "C" size_t pgj_oc_ws_bytes(int n) {
  const int64_t N = int64_t(n) * n * n;
  return align256(size_t(blocks_of(N)) * 8);
}

extern "C" int pgj_cone_filter(int n, const double* x, const int32_t* offsets, const double* weights, int m,
                               double* y, const double* bounds, int conditional, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && offsets && weights && y && m >= 1, "invalid cone filter arguments");
  PGJ_REQUIRE(!conditional || bounds, "conditional filtering needs bounds");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_filter_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), x, offsets, weights, m,
                     n, y, bounds, conditional);
  PGJ_LAUNCHED("cone_filter");
  return PGJ_OK;
}

extern "C" int pgj_cone_project(int n, const double* t, const double* hs, double* ph, double* dp, double* a,
                                const double* bounds, double beta, double eta, double emin, int conditional,
                                double* ws, void* stream) {
  PGJ_REQUIRE(n >= 2 && t && hs && ph && dp && a, "invalid projection arguments");
  PGJ_REQUIRE(!conditional || bounds, "conditional projection needs bounds");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_project_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), t, hs, ph, dp, a, bounds,
                     N, beta, eta, emin, conditional, ws);
  PGJ_LAUNCHED("cone_project");
  return PGJ_OK;
}

extern "C" int pgj_cone_sensitivity(int n, const double* dp, const double* ph, const double* energy, const double* hs,
                                    double emin, double* gin, double* dvin, void* stream) {
  PGJ_REQUIRE(n >= 2 && dp && ph && energy && hs && gin && dvin, "invalid sensitivity arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_prepare_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), dp, ph, energy, hs, emin,
                     N, gin, dvin);
  PGJ_LAUNCHED("cone_prepare");
  return PGJ_OK;
}

extern "C" int pgj_cone_ratio(int n, double* g, const double* dv, double* ratio, double* bounds, void* stream) {
  PGJ_REQUIRE(n >= 2 && g && dv && ratio && bounds, "invalid ratio arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_ratio_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), g, dv, N, ratio, bounds);
  PGJ_LAUNCHED("cone_ratio");
  return PGJ_OK;
}

extern "C" int pgj_cone_candidate(int n, const double* x, const double* ratio, const double* bounds, double move,
                                  double* y, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && ratio && bounds && y, "invalid candidate arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_candidate_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), x, ratio, bounds, move,
                     y, N);
  PGJ_LAUNCHED("cone_candidate");
  return PGJ_OK;
}

extern "C" int pgj_cone_bisect(int n, const double* ws, double* bounds, double volume, void* stream) {
  PGJ_REQUIRE(n >= 2 && ws && bounds, "invalid bisection arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(cone_bisect_kernel, dim3(1), dim3(64), 0, as_stream(stream), ws, blocks_of(N), N, bounds, volume);
  PGJ_LAUNCHED("cone_bisect");
  return PGJ_OK;
}

extern "C" int pgj_absmax_diff(int n, const double* a, const double* b, double* ws, double* out, void* stream) {
  PGJ_REQUIRE(n >= 2 && a && b && ws && out, "invalid absmax arguments");
  const int64_t N = int64_t(n) * n * n;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(absmax_partials, dim3(blocks_of(N)), dim3(256), 0, s, a, b, N, ws);
  PGJ_LAUNCHED("absmax_partials");
  hipLaunchKernelGGL(absmax_finish, dim3(1), dim3(64), 0, s, ws, blocks_of(N), out);
  PGJ_LAUNCHED("absmax_finish");
  return PGJ_OK;
}

extern "C" int pgj_gauss_filter(int n, const double* x, const double* weights, int radius, double* tmp1, double* tmp2,
                                double* y, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && weights && tmp1 && tmp2 && y && radius >= 0 && radius <= 4 * n,
              "invalid gaussian filter arguments");
  const int64_t N = int64_t(n) * n * n;
  hipStream_t s = as_stream(stream);
  if (pgj_gauss_fused(n, radius) && tmp1 != y) {   // y may alias x or tmp1, as before
    hipLaunchKernelGGL(gauss_z_kernel<false>, dim3(gauss_columns(n)), dim3(256), size_t(n) * kGaussCols * 8, s, x,
                       nullptr, 0.0, 0.0, nullptr, nullptr, 0, nullptr, weights, radius, n, nullptr, tmp1);
    hipLaunchKernelGGL(gauss_yx_kernel<false>, dim3(gauss_strips(n), n), dim3(256), gauss_lds(n, radius), s, tmp1,
                       weights, radius, n, gauss_inv(n), 0.0, y, nullptr);
    PGJ_LAUNCHED("gauss_filter");
    return PGJ_OK;
  }
  hipLaunchKernelGGL(gauss_axis_kernel, dim3(blocks_of(N)), dim3(256), 0, s, x, weights, radius, n, 0, tmp1);
  hipLaunchKernelGGL(gauss_axis_kernel, dim3(blocks_of(N)), dim3(256), 0, s, tmp1, weights, radius, n, 1, tmp2);
  hipLaunchKernelGGL(gauss_axis_kernel, dim3(blocks_of(N)), dim3(256), 0, s, tmp2, weights, radius, n, 2, y);
  PGJ_LAUNCHED("gauss_axis");
  return PGJ_OK;
}

extern "C" int pgj_gauss_project(int n, const double* t, double beta, double* ph, double* dp, double* a, double emin,
                                 double* ws, void* stream) {
  PGJ_REQUIRE(n >= 2 && t && ph && dp && a, "invalid projection arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(gauss_project_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), t, beta, ph, dp, a, N,
                     emin, ws);
  PGJ_LAUNCHED("gauss_project");
  return PGJ_OK;
}

extern "C" int pgj_gauss_sensitivity(int n, const double* dp, const double* ph, const double* energy, double emin,
                                     double penal, double* gin, void* stream) {
  PGJ_REQUIRE(n >= 2 && dp && ph && energy && gin, "invalid sensitivity arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(gauss_prepare_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), dp, ph, energy, emin,
                     penal, N, gin);
  PGJ_LAUNCHED("gauss_prepare");
  return PGJ_OK;
}

extern "C" int pgj_gauss_ratio(int n, const double* g, const double* dv, double* ratio, double* ws, double* bounds,
                               void* stream) {
  PGJ_REQUIRE(n >= 2 && g && dv && ratio && ws && bounds, "invalid ratio arguments");
  const int64_t N = int64_t(n) * n * n;
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(gauss_ratio_kernel, dim3(blocks_of(N)), dim3(256), 0, s, g, dv, N, ratio, ws);
  PGJ_LAUNCHED("gauss_ratio");
  hipLaunchKernelGGL(gauss_bounds_kernel, dim3(1), dim3(64), 0, s, ws, blocks_of(N), bounds);
  PGJ_LAUNCHED("gauss_bounds");
  return PGJ_OK;
}

extern "C" int pgj_gauss_candidate(int n, const double* x, const double* ratio, const double* bounds, double move,
                                   double* y, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && ratio && bounds && y, "invalid candidate arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(gauss_candidate_kernel, dim3(blocks_of(N)), dim3(256), 0, as_stream(stream), x, ratio, bounds,
                     move, y, N);
  PGJ_LAUNCHED("gauss_candidate");
  return PGJ_OK;
}

extern "C" int pgj_gauss_bisect(int n, const double* ws, double* bounds, double volume, void* stream) {
  PGJ_REQUIRE(n >= 2 && ws && bounds, "invalid bisection arguments");
  const int64_t N = int64_t(n) * n * n;
  hipLaunchKernelGGL(gauss_bisect_kernel, dim3(1), dim3(64), 0, as_stream(stream), ws, blocks_of(N), N, bounds, volume);
  PGJ_LAUNCHED("gauss_bisect");
  return PGJ_OK;
}

// ------------------------------------------------------------- fused entries
namespace {
dim3 cone_grid(int n) { return dim3((n + kTX - 1) / kTX, (n + kTY - 1) / kTY, (n + kTZ - 1) / kTZ); }
int cone_blocks(int n) {
  const dim3 g = cone_grid(n);
  return int(g.x * g.y * g.z);
}
ConeProjection cone_projection(double beta, double eta) {
  const double te = std::tanh(beta * eta);
  return {beta, eta, te, te + std::tanh(beta * (1 - eta))};
}
#define PGJ_CONE_REACH(CALL)      \
  switch (reach) {                \
    case 0: case 1: CALL(1); break; \
    case 2: CALL(2); break;       \
    default: CALL(3); break;      \
  }
#define PGJ_REQUIRE_REACH                                                                                         \
  PGJ_REQUIRE(reach >= 0 && reach <= kConeReach, "the fused cone passes take a reach of 0..%d planes, got %d", \
              kConeReach, reach)

}  // namespace

extern "C" int pgj_cone_max_reach(void) { return kConeReach; }

extern "C" int pgj_cone_physical(int n, const double* x, const int32_t* offsets, const double* weights, int m, int reach,
                                 const double* hs, double beta, double eta, double emin, double* t, double* ph,
                                 double* dp, double* a, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && offsets && weights && m >= 1 && hs && t && ph && dp && a, "invalid cone arguments");
  PGJ_REQUIRE_REACH;
  const ConeStencil c{n, m, offsets, weights};
#define CALL(R)                                                                                                    \
  hipLaunchKernelGGL(cone_physical_kernel<R>, cone_grid(n), dim3(kConeThreads), 0, as_stream(stream), c, x, hs, \
                     cone_projection(beta, eta), emin, t, ph, dp, a)
  PGJ_CONE_REACH(CALL)
#undef CALL
  PGJ_LAUNCHED("cone_physical");
  return PGJ_OK;
}

extern "C" int pgj_cone_gradient(int n, const double* dp, const double* ph, const double* energy, const double* hs,
                                 const int32_t* offsets, const double* weights, int m, int reach, double emin, double* g,
                                 double* dv, double* ratio, double* root, double* bounds, void* stream) {
  PGJ_REQUIRE(n >= 2 && dp && ph && energy && hs && offsets && weights && m >= 1 && g && dv && ratio && root && bounds,
              "invalid cone gradient arguments");
  PGJ_REQUIRE_REACH;
  const ConeStencil c{n, m, offsets, weights};
#define CALL(R)                                                                                                      \
  hipLaunchKernelGGL(cone_gradient_kernel<R>, cone_grid(n), dim3(kConeThreads), 0, as_stream(stream), c, dp, ph, energy, hs, emin, \
                     g, dv, ratio, reinterpret_cast<double2*>(root), bounds)
  PGJ_CONE_REACH(CALL)
#undef CALL
  PGJ_LAUNCHED("cone_gradient");
  return PGJ_OK;
}

extern "C" size_t pgj_cone_rounds_ws_bytes(int n) { return n < 2 ? 0 : align256((size_t(cone_blocks(n)) * 2 + 8) * 8); }

extern "C" int pgj_cone_rounds(int n, const double* x, const double* root, const int32_t* offsets,
                               const double* weights, int m, int reach, const double* hs, double beta, double eta,
                               double move, double volume, int rounds, double* y, double* bounds, double* ws,
                               void* stream) {
  PGJ_REQUIRE(n >= 2 && x && root && offsets && weights && m >= 1 && hs && y && bounds && ws && rounds >= 1,
              "invalid cone bisection arguments");
  PGJ_REQUIRE_REACH;
  const ConeStencil c{n, m, offsets, weights};
  hipStream_t s = as_stream(stream);
  // two sets of bounds and of volume partials, by parity of the round
  const int nblk = cone_blocks(n);
  const ConeProjection pr = cone_projection(beta, eta);
  const double floor03 = std::pow(1e-10, 0.3);
  double* b[2] = {ws, ws + 4};
  double* v[2] = {ws + 8, ws + 8 + nblk};
  for (int k = 0; k < rounds; ++k) {
    const double* in = k == 0 ? bounds : b[(k - 1) & 1];
    const double* vprev = k == 0 ? nullptr : v[(k - 1) & 1];
#define CALL(R)                                                                                                     \
  hipLaunchKernelGGL(cone_round_kernel<R>, cone_grid(n), dim3(kConeThreads), 0, s, c, x, \
                     reinterpret_cast<const double2*>(root), hs, pr, floor03, move, volume, in, vprev, b[k & 1],      \
                     v[k & 1], y)
    PGJ_CONE_REACH(CALL)
#undef CALL
    PGJ_LAUNCHED("cone_round");
  }
  hipLaunchKernelGGL(cone_rounds_finish, dim3(1), dim3(64), 0, s, b[(rounds - 1) & 1], v[(rounds - 1) & 1], nblk,
                     int64_t(n) * n * n, volume, bounds);
  PGJ_LAUNCHED("cone_rounds_finish");
  return PGJ_OK;
}

extern "C" int pgj_gauss_fused(int n, int radius) { return n >= 2 && radius >= 0 && gauss_fused(n, radius) ? 1 : 0; }

extern "C" size_t pgj_gauss_rounds_ws_bytes(int n) {
  return n < 2 ? 0 : align256((size_t(gauss_strips(n)) * n + 4) * 8);
}

extern "C" int pgj_gauss_rounds(int n, const double* x, const double* ratio, const double* weights, int radius,
                                double* tmp, double beta, double move, double volume, int rounds, double* y,
                                double* bounds, double* ws, void* stream) {
  PGJ_REQUIRE(n >= 2 && x && ratio && weights && radius >= 0 && tmp && y && bounds && ws && rounds >= 1,
              "invalid gaussian bisection arguments");
  PGJ_REQUIRE(gauss_fused(n, radius), "the fused gaussian passes do not take n = %d with radius %d", n, radius);
  hipStream_t s = as_stream(stream);
  const int nblk = gauss_strips(n) * n;
  double* b[2] = {ws, ws + 2};
  double* v = ws + 4;   // written by a round's second launch, read by the next round's first
  for (int k = 0; k < rounds; ++k) {
    hipLaunchKernelGGL(gauss_z_kernel<true>, dim3(gauss_columns(n)), dim3(256), size_t(n) * kGaussCols * 8, s, x, ratio,
                       move, volume, k == 0 ? bounds : b[(k - 1) & 1], k == 0 ? nullptr : v, nblk, b[k & 1], weights,
                       radius, n, y, tmp);
    hipLaunchKernelGGL(gauss_yx_kernel<true>, dim3(gauss_strips(n), n), dim3(256), gauss_lds(n, radius), s, tmp, weights,
                       radius, n, gauss_inv(n), beta, nullptr, v);
    PGJ_LAUNCHED("gauss_round");
  }
  hipLaunchKernelGGL(gauss_rounds_finish, dim3(1), dim3(64), 0, s, b[(rounds - 1) & 1], v, nblk, int64_t(n) * n * n,
                     volume, bounds);
  PGJ_LAUNCHED("gauss_rounds_finish");
  return PGJ_OK;
}
