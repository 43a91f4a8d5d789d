// Hand-written FP64 3-D R2C/C2R FFT for runtime shapes (LDS Stockham, radices
// 2..10) with the FI Green symbol fused into the z pass, and the pre/post
// scaling, projection and PCG vector updates fused into the xy passes.
//
// Data path per load (spectrum layout S[l][c][kz][ky][kx], kx < nx/2+1):
//   fxy  : per z-plane and component, v = s*r (PCG: r -= alpha q first);
//          x-R2C (two reals per complex line + split), y-FFT; write S.
//   fz   : per chunk of (ky, kx) columns, z-FFT, v^ -= mean(r) s^ (projection P),
//          w^ = G v^, Parseval partials of v.w and s.w, inverse z-FFT.
//   fxyi : per z-plane and component, inverse y-FFT, x-C2R, z = s*w - mean(s*w)
//          (PCG: written as the next direction z + beta p; u += alpha p).
//
// What bounds these passes on small and middle grids is the chain of dependent steps in a block, not bytes: with
// block-wide stages (2 barriers each, radices 4/2/3/5/7), run-time divisions in every index (64-bit ones in the loops)
// and twiddles from global memory the three launches at 40^3, three loads, took 48 + 33 + 47 us (now 14.6 + 15.3 + 14.1), and
// the preconditioner of 45x60x50, three loads, 153 us (now 47). Here a wavefront
// carries whole lines through all stages without a barrier (AxisPlan: 2 stages for nearly every length up to 100), the
// divisions are multiplications by constants of the plan, and the twiddles are in LDS.
#include <cmath>

#include "fft_kernels.h"
#include "stockham.h"

namespace pgj {

// LDS reads and writes of one wavefront, in program order for all its lanes.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One in-place Stockham stage of the line at `L` (elements es apart), by the lanes j0 of its group.
template <int R, bool INV>
__device__ __forceinline__ void line_stage(double2* L, int es, bool on, int j0, int G, const AxisPlan::Stage& st,
                                           const double2* tw, int step) {
  constexpr int NB = R == 3 ? 2 : 1;  // only n / 3 can pass the 64 lanes of a group (n = 243)
  double2 v[NB][R];
  int out[NB];
  const int Ns = st.Ns, rd = st.nb * es;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int j = j0 + i * G;
    out[i] = -1;
    if (on && j < st.nb) {
      const int q = int((unsigned(j) * st.mNs) >> 16), k = j - q * Ns;
      out[i] = (q * Ns * R + k) * es;
      const double2* p = L + j * es;
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = p[r * rd];
      if (Ns > 1) {
        const int t = k * st.tws * step;
#pragma unroll
        for (int r = 1; r < R; ++r) v[i][r] = cmul(v[i][r], twiddle<INV>(tw, r * t, 1));
      }
    }
  }
  wave_fence();
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (out[i] >= 0) {
      dft<R, INV>(v[i], tw, 0, 0);
      double2* p = L + out[i];
#pragma unroll
      for (int r = 0; r < R; ++r) p[r * Ns * es] = v[i][r];
    }
  }
  wave_fence();
}

// All stages of one line per group of lanes.
template <bool INV>
__device__ __forceinline__ void line_fft(double2* L, int es, bool on, int j0, const AxisPlan& a, const double2* tw,
                                         int step) {
#pragma unroll 1
  for (int s = 0; s < a.count; ++s) {
    const AxisPlan::Stage& st = a.st[s];
    switch (st.R) {
      case 2: line_stage<2, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 3: line_stage<3, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 4: line_stage<4, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 5: line_stage<5, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 6: line_stage<6, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 7: line_stage<7, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 8: line_stage<8, INV>(L, es, on, j0, a.G, st, tw, step); break;
      case 9: line_stage<9, INV>(L, es, on, j0, a.G, st, tw, step); break;
      default: line_stage<10, INV>(L, es, on, j0, a.G, st, tw, step); break;
    }
  }
}

// Place of a lane in its wavefront's group of lines: line `line` of the group (on: it carries one) and lane j0 of that
// line. FAST: consecutive lanes take consecutive lines (columns in LDS), else consecutive elements (rows).
template <bool FAST>
struct LanePlace {
  int line, j0;
  bool on;
  __device__ __forceinline__ explicit LanePlace(const AxisPlan& a) {
    const unsigned lane = threadIdx.x & 63;
    if (FAST) {
      j0 = int((lane * a.mL) >> 16);
      line = int(lane) - j0 * a.lpw;
      on = j0 < a.G;
    } else {
      line = int((lane * a.mG) >> 16);
      j0 = int(lane) - line * a.G;
      on = line < a.lpw;
    }
  }
};

// Transforms of the columns 0..ncol of a plane in LDS (rows rs apart).
template <bool INV>
__device__ __forceinline__ void column_ffts(double2* plane, int ncol, int rs, const AxisPlan& a, const double2* tw) {
  const LanePlace<true> at(a);
  const int wave = threadIdx.x >> 6, step = (blockDim.x >> 6) * a.lpw;
  for (int l0 = wave * a.lpw; l0 < ncol; l0 += step) {
    const int line = l0 + at.line;
    line_fft<INV>(plane + line, rs, at.on && line < ncol, at.j0, a, tw, 1);
  }
}

__device__ __forceinline__ double reduce_pr_sum(const FFTArgs& A, int l, int c) {
  // sum over planes of the per-plane component sums (fixed order, every lane identical)
  return wave_reduce_partials(A.pr + (int64_t(l) * A.nz * 3 + c) * 2 + 1, A.nz, 6);
}

// Plane z and component c of a block of the xy passes. The three components of a plane run on one XCD (block ids 8
// apart), because in the node-interleaved layout they share every line of r, s and z.
__device__ __forceinline__ bool plane_of_block(int nz, int& z, int& c) {
  const int id = blockIdx.x, group = id / 24, rem = id % 24;
  c = rem / 8;
  z = group * 8 + rem % 8;
  return z < nz;
}

// Copies the twiddle tables of the xy passes to LDS, x before y.
__device__ __forceinline__ void plane_twiddles(const FFTArgs& A, double2* lds) {
  for (int i = threadIdx.x; i < A.nx; i += blockDim.x) lds[i] = A.twx[i];
  for (int i = threadIdx.x; i < A.ny; i += blockDim.x) lds[A.nx + i] = A.twy[i];
}

constexpr int kRedDoubles = 32;  // LDS scratch of the block sums, ahead of the plane
constexpr int kPlaneUnroll = 4;  // values of a plane a thread loads before it uses the first

// --------------------------------------------------------------- forward xy
template <int MODE>
__global__ __launch_bounds__(512) void fxy_kernel(FFTArgs A) {
  extern __shared__ double smem[];
  const FFTGeom& f = A.f;
  int z, c;
  if (!plane_of_block(A.nz, z, c)) return;
  const int l = blockIdx.z, T = blockDim.x;
  if (MODE == kFxyPCG && !A.st.active[l]) return;
  const int nx = A.nx, ny = A.ny, pn = nx * ny, rs = f.rs;
  double* red = smem;
  double2* plane = reinterpret_cast<double2*>(smem + kRedDoubles);
  double2 *twx = plane + ny * rs, *twy = twx + nx;
  plane_twiddles(A, twx);

  // 1. load (and update) the plane; pack reals two per complex along x.
  const int ns = A.soa ? 1 : 3;
  const int dl = design_of(l, A.group);
  const int64_t p0 = int64_t(z) * pn;
  const int64_t off = A.soa ? (int64_t(l) * 3 + c) * A.N + p0 : (int64_t(l) * A.N + p0) * 3 + c;
  const int64_t soff = A.soa ? (int64_t(dl) * 3 + c) * A.N + p0 : (int64_t(dl) * A.N + p0) * 3 + c;
  const double* sp = A.s ? A.s + soff : nullptr;
  const double* in = MODE == kFxyPCG ? A.r + off : A.rin + off;
  const double* qp = A.q + off;
  double* rp = A.r + off;
  const unsigned mx = f.mnx;
  const bool even = (nx % 2) == 0;
  double alpha = 0.0, sums[2] = {0.0, 0.0};
  for (int e0 = 0; e0 < pn; e0 += kPlaneUnroll * T) {
    double vr[kPlaneUnroll], vq[kPlaneUnroll], vs[kPlaneUnroll];
#pragma unroll
    for (int i = 0; i < kPlaneUnroll; ++i) {
      const int e = min(e0 + i * T + int(threadIdx.x), pn - 1) * ns;
      if (MODE != kFxyScale) vr[i] = in[e];
      if (MODE == kFxyPCG) vq[i] = qp[e];
      vs[i] = sp ? sp[e] : 1.0;
    }
    if (MODE == kFxyPCG && e0 == 0) {
      // the step length is reduced while the first loads are in flight
      double pq, rz;
      wave_reduce_partials_2(A.ppq + int64_t(l) * A.ppq_stride, A.ppq_count, 1, A.pg + int64_t(l) * f.nkb * ny * 4,
                             A.zslots, 4, pq, rz);
      const bool valid = isfinite(pq) && pq > 0.0 && isfinite(rz) && rz > 0.0;
      alpha = valid ? rz / pq : 0.0;
      if (threadIdx.x == 0 && blockIdx.x == 0) {
        A.st.rz[l] = rz;
        A.st.alpha[l] = alpha;
        A.st.valid[l] = valid;
        A.st.first[l] = 0;
      }
    }
#pragma unroll
    for (int i = 0; i < kPlaneUnroll; ++i) {
      const int e = e0 + i * T + int(threadIdx.x);
      if (e < pn) {
        double val = vs[i];
        if (MODE != kFxyScale) {
          double rn = vr[i];
          if (MODE == kFxyPCG) {
            rn = fma(-alpha, vq[i], rn);
            rp[e * ns] = rn;
          }
          sums[0] = fma(rn, rn, sums[0]);
          sums[1] += rn;
          val = sp ? val * rn : rn;
        }
        const int y = int(__umulhi(unsigned(e), mx)), x = e - y * nx;
        double2* row = plane + y * rs;
        if (even) reinterpret_cast<double*>(row)[x] = val;
        else row[x] = c2(val, 0.0);
      }
    }
  }
  if (MODE != kFxyScale) {
    block_sums<2>(sums, red);
    if (threadIdx.x == 0) {
      double* p = A.pr + ((int64_t(l) * A.nz + z) * 3 + c) * 2;
      p[0] = sums[0];
      p[1] = sums[1];
    }
  }
  __syncthreads();
  // 2. x transform of every row (complex length M) and the split of the packed spectrum into the half spectrum of the
  // real row, by the row's own lanes
  {
    const AxisPlan& a = f.px;
    const LanePlace<false> at(a);
    const int M = f.M, half = M / 2, step = (T >> 6) * a.lpw, wstep = even ? 2 : 1;
    for (int l0 = (threadIdx.x >> 6) * a.lpw; l0 < ny; l0 += step) {
      const int row = l0 + at.line;
      const bool on = at.on && row < ny;
      double2* L = plane + row * rs;
      line_fft<false>(L, 1, on, at.j0, a, twx, wstep);
      if (even && on) {
        for (int k = at.j0; k <= half; k += a.G) {
          const double2 zk = L[k], zm = L[k == 0 ? 0 : M - k];
          const double2 E = c2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
          const double2 O = c2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
          const double2 wo = cmul(twx[k], O);
          L[k] = cadd(E, wo);
          if (M - k != k) L[M - k] = conjd(csub(E, wo));
        }
      }
    }
  }
  __syncthreads();
  // 3. y transform of every kx column.
  column_ffts<false>(plane, f.nkx, rs, f.py, twy);
  __syncthreads();
  // 4. write the half spectrum.
  double2* out = A.spec + ((int64_t(l) * 3 + c) * A.nz + z) * (ny * f.nkx);
  const unsigned mk = f.mnkx;
  const int total = ny * f.nkx, pad = rs - f.nkx;
  for (int e = threadIdx.x; e < total; e += T) out[e] = plane[e + (pad ? int(__umulhi(unsigned(e), mk)) * pad : 0)];
}

// ---------------------------------------------------------------- z + Green
// A block transforms C consecutive columns (ky, kx) of the three components, all in LDS [c][z][column]. C = 16 fills
// two lines of every row it reads; 8 and 4 spread small grids over the CUs (runtime_chunk).
template <int MODE, int C>
__global__ __launch_bounds__(512) void fz_kernel(FFTArgs A) {
  extern __shared__ double smem[];
  const FFTGeom& f = A.f;
  const int l = blockIdx.z, T = blockDim.x;
  const int nz = A.nz, nzc = nz * C, pl = A.ny * f.nkx;
  const int f0 = blockIdx.x * C, ncol = min(C, pl - f0);
  const bool lead = threadIdx.x == 0 && blockIdx.x == 0;
  double* red = smem;
  double2* cols = reinterpret_cast<double2*>(smem + kRedDoubles);
  double2* tw = cols + 3 * nzc;
  double2* S = A.spec + int64_t(l) * 3 * f.nf + f0;
  if (MODE == kFzPCG && !A.st.active[l]) {
    // an inactive load stays inactive: the test below with active = false
    if (lead) {
      A.st.active_next[l] = 0;
      A.st.it_next[l] = A.st.it[l];
      A.st.bad_next[l] = A.st.bad[l];
      A.st.stopped[l] = 0;
    }
    return;
  }
  // the columns and twiddles go to LDS first; the test below runs while they are in flight
  for (int e = threadIdx.x; e < 3 * nzc; e += T) {
    const int col = e % C, row = e / C;
    cols[e] = col < ncol ? S[int64_t(row) * pl + col] : c2(0.0, 0.0);
  }
  for (int i = threadIdx.x; i < nz; i += T) tw[i] = A.twz[i];
  double mean[3] = {0.0, 0.0, 0.0};
  if (MODE == kFzInit || MODE == kFzPCG) {
    // one pass over the per-plane partials (|r|^2 and the component sums of r)
    const int lane = threadIdx.x & 63;
    double v = 0.0, vm[3] = {0.0, 0.0, 0.0};
    for (int i = lane; i < nz; i += 64) {
      const double* p = A.pr + (int64_t(l) * nz + i) * 6;
      v += (p[0] + p[2]) + p[4];
      vm[0] += p[1];
      vm[1] += p[3];
      vm[2] += p[5];
    }
    const double res2 = wave_sum(v);
    if (A.shat)
      for (int c = 0; c < 3; ++c) mean[c] = wave_sum(vm[c]) / double(A.N);
    bool act;
    if (MODE == kFzInit) {
      act = res2 > A.st.target2[l] && A.st.it[l] < A.st.cap[l] && !A.st.bad[l];
      if (lead) {
        A.st.active_next[l] = act;
        A.st.it_next[l] = A.st.it[l];
        A.st.bad_next[l] = A.st.bad[l];
        A.st.first[l] = 1;
        A.st.stopped[l] = 0;
      }
    } else {
      const bool valid = A.st.valid[l] != 0;  // set by the forward pass of this iteration
      const bool finite = isfinite(res2);
      const int64_t it = A.st.it[l] + 1;
      act = valid && finite && res2 > A.st.target2[l] && it < A.st.cap[l];
      if (lead) {
        A.st.active_next[l] = act;
        A.st.it_next[l] = it;
        A.st.bad_next[l] = A.st.bad[l] || !valid || !finite;
        A.st.stopped[l] = !act;
      }
    }
    if (!act) return;
  } else if (MODE != kFzScale && A.shat) {
    for (int c = 0; c < 3; ++c) mean[c] = reduce_pr_sum(A, l, c) / double(A.N);
  }
  __syncthreads();
  const AxisPlan& a = f.pz;
  const LanePlace<true> at(a);
  const int wave0 = (threadIdx.x >> 6) * a.lpw, step = (T >> 6) * a.lpw;
  for (int l0 = wave0; l0 < 3 * C; l0 += step) {
    const int line = l0 + at.line;
    line_fft<false>(cols + line / C * nzc + line % C, C, at.on && line < 3 * C, at.j0, a, tw, 1);
  }
  __syncthreads();
  if (MODE != kFzScale) {
    // per frequency: projection correction, Green multiply, Parseval partials
    double sums[4] = {0.0, 0.0, 0.0, 0.0};  // r.z, s.w of the three components
    const unsigned mk = f.mnkx;
    for (int e = threadIdx.x; e < nzc; e += T) {
      const int col = e % C, zz = e / C;
      if (col >= ncol) continue;
      const int fk = f0 + col, kx = fk - int(__umulhi(unsigned(fk), mk)) * f.nkx;
      const int64_t fidx = int64_t(zz) * pl + fk;
      double g[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) g[i] = A.sym[i * f.nf + fidx];
      double2 v[3], sh[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = cols[c * nzc + e];
      if (A.shat) {
#pragma unroll
        for (int c = 0; c < 3; ++c) sh[c] = A.shat[(int64_t(design_of(l, A.group)) * 3 + c) * f.nf + fidx];
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = c2(fma(-mean[c], sh[c].x, v[c].x), fma(-mean[c], sh[c].y, v[c].y));
      }
      double2 w[3];
      w[0] = c2(g[0] * v[0].x + g[3] * v[1].x + g[4] * v[2].x, g[0] * v[0].y + g[3] * v[1].y + g[4] * v[2].y);
      w[1] = c2(g[3] * v[0].x + g[1] * v[1].x + g[5] * v[2].x, g[3] * v[0].y + g[1] * v[1].y + g[5] * v[2].y);
      w[2] = c2(g[4] * v[0].x + g[5] * v[1].x + g[2] * v[2].x, g[4] * v[0].y + g[5] * v[1].y + g[2] * v[2].y);
      const double wgt = (kx == 0 || (A.nx % 2 == 0 && kx == A.nx / 2)) ? 1.0 : 2.0;
      double t = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) t += v[c].x * w[c].x + v[c].y * w[c].y;
      sums[0] = fma(wgt, t, sums[0]);
      if (A.shat)
#pragma unroll
        for (int c = 0; c < 3; ++c) sums[1 + c] = fma(wgt, sh[c].x * w[c].x + sh[c].y * w[c].y, sums[1 + c]);
#pragma unroll
      for (int c = 0; c < 3; ++c) cols[c * nzc + e] = w[c];
    }
    block_sums<4>(sums, red);
    if (threadIdx.x == 0) {
      double* pg = A.pg + (int64_t(l) * f.nkb * A.ny + blockIdx.x) * 4;
      for (int i = 0; i < 4; ++i) pg[i] = sums[i];
    }
    __syncthreads();
    for (int l0 = wave0; l0 < 3 * C; l0 += step) {
      const int line = l0 + at.line;
      line_fft<true>(cols + line / C * nzc + line % C, C, at.on && line < 3 * C, at.j0, a, tw, 1);
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < 3 * nzc; e += T) {
    const int col = e % C, row = e / C;
    if (col < ncol) S[int64_t(row) * pl + col] = cols[e];
  }
}

// --------------------------------------------------------------- inverse xy
template <int MODE>
__global__ __launch_bounds__(512) void fxyi_kernel(FFTArgs A) {
  extern __shared__ double smem[];
  const FFTGeom& f = A.f;
  int z, c;
  if (!plane_of_block(A.nz, z, c)) return;
  const int l = blockIdx.z, T = blockDim.x;
  const int nx = A.nx, ny = A.ny, pn = nx * ny, rs = f.rs, ns = A.soa ? 1 : 3;
  const int dl = design_of(l, A.group);
  const int64_t p0 = int64_t(z) * pn;
  const int64_t off = A.soa ? (int64_t(l) * 3 + c) * A.N + p0 : (int64_t(l) * A.N + p0) * 3 + c;
  const int64_t soff = A.soa ? (int64_t(dl) * 3 + c) * A.N + p0 : (int64_t(dl) * A.N + p0) * 3 + c;
  // PCG: the displacement update u += alpha p of this iteration (alpha from the forward pass)
  const bool move = MODE == kFxyiPCG && A.p != nullptr && A.u != nullptr;
  const double alpha = move ? A.st.alpha[l] : 0.0;
  constexpr bool dir = MODE == kFxyiDir;
  const double* pp = dir ? A.pdir + off : A.p ? A.p + off : nullptr;
  double* up = A.u ? A.u + off : nullptr;
  if (MODE == kFxyiPCG) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
      A.st.active[l] = A.st.active_next[l];
      A.st.it[l] = A.st.it_next[l];
      A.st.bad[l] = A.st.bad_next[l];
    }
    if (!A.st.active_next[l]) {
      // a load stopped by this iteration's test still takes its last displacement update
      if (move && A.st.stopped[l])
        for (int e = threadIdx.x; e < pn; e += T) up[e * ns] = fma(alpha, pp[e * ns], up[e * ns]);
      return;
    }
  }
  double2* plane = reinterpret_cast<double2*>(smem + kRedDoubles);
  double2 *twx = plane + ny * rs, *twy = twx + nx;
  // 1. load the half spectrum of the plane
  const double2* in = A.spec + ((int64_t(l) * 3 + c) * A.nz + z) * (ny * f.nkx);
  const unsigned mk = f.mnkx;
  const int total = ny * f.nkx, pad = rs - f.nkx;
  for (int e = threadIdx.x; e < total; e += T) plane[e + (pad ? int(__umulhi(unsigned(e), mk)) * pad : 0)] = in[e];
  plane_twiddles(A, twx);
  // PCG: the output is the next direction p = z + beta p (z alone right after init)
  double mean = 0.0, beta = 0.0;
  const bool update = dir || (MODE == kFxyiPCG && A.p != nullptr && !A.st.first[l]);
  if (A.shat || update) {
    // one pass: r.z (offset 0) and this component's s.w partials (offset 1 + c)
    const int at[2] = {0, 1 + c};
    double sums[2];
    wave_reduce_partials_n<2>(A.pg + int64_t(l) * f.nkb * ny * 4, at, A.zslots, 4, sums);
    if (A.shat) mean = sums[1] / double(A.N);
    if (dir) {
      beta = sums[0] / fmax(*A.rz_old, 1e-30);
      if (threadIdx.x == 0 && blockIdx.x == 0) *A.rz_out = sums[0];
    } else if (update) {
      const double rz = A.st.rz[l];
      beta = sums[0] / (rz != 0.0 ? rz : 1.0);
    }
  }
  __syncthreads();
  // 2. inverse y transform
  column_ffts<true>(plane, f.nkx, rs, f.py, twy);
  __syncthreads();
  // 3. rebuild the complex line of each real row and transform it, by the row's own lanes
  const bool even = (nx % 2) == 0;
  {
    const AxisPlan& a = f.px;
    const LanePlace<false> at(a);
    const int M = f.M, half = M / 2, step = (T >> 6) * a.lpw;
    for (int l0 = (threadIdx.x >> 6) * a.lpw; l0 < ny; l0 += step) {
      const int row = l0 + at.line;
      const bool on = at.on && row < ny;
      double2* L = plane + row * rs;
      if (even && on) {
        for (int k = at.j0; k <= half; k += a.G) {
          double2 xk = L[k], xm = L[M - k];
          if (k == 0) {
            xk.y = 0.0;
            xm.y = 0.0;
          }
          // Z[k] = (X[k] + conj(X[M-k])) + i (X[k] - conj(X[M-k])) conj(W^k)
          const double2 wk = conjd(twx[k]);
          const double2 e1 = c2(xk.x + xm.x, xk.y - xm.y);
          const double2 o1 = cmul(c2(xk.x - xm.x, xk.y + xm.y), wk);
          if (k != 0 && M - k != k) {
            const double2 wm = conjd(twx[M - k]);
            const double2 e2 = c2(xm.x + xk.x, xm.y - xk.y);
            const double2 o2 = cmul(c2(xm.x - xk.x, xm.y + xk.y), wm);
            L[M - k] = c2(e2.x - o2.y, e2.y + o2.x);
          }
          L[k] = c2(e1.x - o1.y, e1.y + o1.x);
        }
      } else if (on) {
        // odd nx: Hermitian completion of the row
        for (int k = f.nkx + at.j0; k < nx; k += a.G) L[k] = conjd(L[nx - k]);
        if (at.j0 == 0) L[0].y = 0.0;
      }
      wave_fence();
      line_fft<true>(L, 1, on, at.j0, a, twx, even ? 2 : 1);
    }
  }
  __syncthreads();
  // 4. unpack, scale and project; PCG: next direction and displacement update
  const double* sp = A.s ? A.s + soff : nullptr;
  double* zp = (dir ? A.pdir : A.zout) + off;
  const unsigned mx = f.mnx;
  for (int e0 = threadIdx.x; e0 < pn; e0 += kPlaneUnroll * T) {
    double vs[kPlaneUnroll], vp[kPlaneUnroll], vu[kPlaneUnroll];
#pragma unroll
    for (int i = 0; i < kPlaneUnroll; ++i) {
      const int e = min(e0 + i * T, pn - 1) * ns;
      vs[i] = sp ? sp[e] : 1.0;
      vp[i] = update || move ? pp[e] : 0.0;
      vu[i] = move ? up[e] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kPlaneUnroll; ++i) {
      const int e = e0 + i * T;
      if (e < pn) {
        const int y = int(__umulhi(unsigned(e), mx)), x = e - y * nx;
        const double2* row = plane + y * rs;
        const double w = even ? reinterpret_cast<const double*>(row)[x] : row[x].x;
        const double v = sp ? vs[i] * w - mean : w;
        zp[e * ns] = update ? fma(beta, vp[i], v) : v;
        if (move) up[e * ns] = fma(alpha, vp[i], vu[i]);
      }
    }
  }
}

// ----------------------------------------------------------------- plan init
__global__ void plan_twiddles(int nx, int ny, int nz, double2* twx, double2* twy, double2* twz) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  auto w = [](int k, int n) {
    double s, c;
    sincospi(2.0 * double(k) / double(n), &s, &c);
    return c2(c, -s);
  };
  if (i < nx) twx[i] = w(i, nx);
  if (i < ny) twy[i] = w(i, ny);
  if (i < nz) twz[i] = w(i, nz);
}

// FI Green factors at half-spectrum index k: D_ii = 1/(mu t sum(d+v^2) + (lam+mu) t d_i),
// beta = (lam+mu) t / (1 + (lam+mu) t sum v_i^2 D_ii), per-axis v_i; zero at k = 0.
struct FiFactors {
  double inv[3], v[3], beta;
};

__device__ FiFactors fi_factors(int64_t k, int nz, int ny, int nx, double hx, double hy, double hz, double lam,
                                double mu) {
  const int nkx = nx / 2 + 1;
  const int kx = int(k % nkx), ky = int((k / nkx) % ny), kz = int(k / (int64_t(nkx) * ny));
  const int idx[3] = {kx, ky, kz};
  const int n[3] = {nx, ny, nz};
  const double h[3] = {hx, hy, hz};
  FiFactors F;
  double m[3], d[3];
  double t = hx * hy * hz, trace = 0.0;
  for (int i = 0; i < 3; ++i) {
    double s, c;
    sincospi(double(idx[i]) / double(n[i]), &s, &c);
    m[i] = c * c + s * s / 3.0;
    t *= m[i];
    F.v[i] = 2.0 * s * c / (h[i] * m[i]);
    d[i] = 4.0 * (s * s) * (s * s) / (3.0 * h[i] * h[i] * m[i] * m[i]);
    trace += d[i] + F.v[i] * F.v[i];
  }
  trace *= t;
  const double b = (lam + mu) * t;
  double den = 1.0;
  for (int i = 0; i < 3; ++i) {
    F.inv[i] = k == 0 ? 0.0 : 1.0 / (mu * trace + (lam + mu) * t * d[i]);
    den += b * F.v[i] * F.v[i] * F.inv[i];
  }
  F.beta = k == 0 ? 0.0 : b / den;
  return F;
}

// Dense FI Green symbol: G = (D - beta (Dv)(Dv)^T)/N.
__global__ void plan_symbol(int nz, int ny, int nx, double hx, double hy, double hz, double lam, double mu,
                            double* sym) {
  const int64_t nf = int64_t(nz) * ny * (nx / 2 + 1);
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= nf) return;
  const FiFactors F = fi_factors(k, nz, ny, nx, hx, hy, hz, lam, mu);
  const double beta = F.beta;
  const double invN = 1.0 / (double(nx) * ny * nz);
  double w[3];
  for (int i = 0; i < 3; ++i) w[i] = F.inv[i] * F.v[i];
  sym[k] = (F.inv[0] - beta * w[0] * w[0]) * invN;
  sym[nf + k] = (F.inv[1] - beta * w[1] * w[1]) * invN;
  sym[2 * nf + k] = (F.inv[2] - beta * w[2] * w[2]) * invN;
  sym[3 * nf + k] = -beta * w[0] * w[1] * invN;
  sym[4 * nf + k] = -beta * w[0] * w[2] * invN;
  sym[5 * nf + k] = -beta * w[1] * w[2] * invN;
}

// The factored form (D_00, D_11, D_22, beta) per k, unnormalised, and the per-axis
// v tables (x over nx/2+1, then y, then z).
__global__ void fi_coeff_kernel(int nz, int ny, int nx, double hx, double hy, double hz, double lam, double mu,
                                double* out4, double* vtab) {
  const int nkx = nx / 2 + 1;
  const int64_t nf = int64_t(nz) * ny * nkx;
  const int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k >= nf) return;
  const FiFactors F = fi_factors(k, nz, ny, nx, hx, hy, hz, lam, mu);
  for (int i = 0; i < 3; ++i) out4[i * nf + k] = F.inv[i];
  out4[3 * nf + k] = F.beta;
  if (vtab) {
    const int kx = int(k % nkx), ky = int((k / nkx) % ny), kz = int(k / (int64_t(nkx) * ny));
    if (ky == 0 && kz == 0) vtab[kx] = F.v[0];
    if (kx == 0 && kz == 0) vtab[nkx + ky] = F.v[1];
    if (kx == 0 && ky == 0) vtab[nkx + ny + kz] = F.v[2];
  }
}

// ------------------------------------------------------------------ launchers
FFTArgs fft_args(const pgj_grid& g, const void* plan) {
  FFTArgs A{};
  A.nz = g.nz; A.ny = g.ny; A.nx = g.nx;
  A.N = int64_t(g.nx) * g.ny * g.nz;
  A.f = fft_geom(g);
  PlanLayout pl = plan_layout(g);
  const char* b = static_cast<const char*>(plan);
  A.twx = reinterpret_cast<const double2*>(b + pl.tw_x);
  A.twy = reinterpret_cast<const double2*>(b + pl.tw_y);
  A.twz = reinterpret_cast<const double2*>(b + pl.tw_z);
  A.sym = reinterpret_cast<const double*>(b + pl.sym);
  return A;
}

int check_fft(const pgj_grid* g) {
  PGJ_REQUIRE(g != nullptr, "null grid");
  FFTGeom f = fft_geom(*g);
  PGJ_REQUIRE(f.valid, "unsupported FFT grid (%d,%d,%d): axis lengths must be 2..256 with factors 2,3,5,7",
              g->nz, g->ny, g->nx);
  return PGJ_OK;
}

// Kernels using more than 64 KiB of dynamic LDS must opt in once.
template <typename K>
int allow_lds(K kernel, size_t bytes) {
  if (bytes <= 65536) return PGJ_OK;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
  if (e != hipSuccess) {
    set_error("cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
    return PGJ_ERR_HIP;
  }
  return PGJ_OK;
}

#define PGJ_RUNTIME_FFT(A)                                                                              \
  PGJ_REQUIRE((A).f.runtime_ok, "grid (%d,%d,%d) has only the compile-time resident FFT path", (A).nz, (A).ny, \
              (A).nx)

// Threads of a block whose transforms carry `lines` lines of plan `a`: one round of wavefronts, 256 to 512 threads.
inline int line_threads(const AxisPlan& a, int lines) {
  const int waves = (lines + a.lpw - 1) / a.lpw;
  return 64 * std::min(8, std::max(4, waves));
}

struct PlaneLaunch {
  dim3 grid;
  int threads;
  size_t lds;  // below 148 KB: the supported planes hold at most 8192 + ny values (fft_geom)
};

inline PlaneLaunch plane_launch(const FFTArgs& A, int L) {
  PlaneLaunch p;
  p.grid = dim3(unsigned((A.nz + 7) / 8 * 24), 1, unsigned(L));
  p.threads = std::max(line_threads(A.f.px, A.ny), line_threads(A.f.py, A.f.nkx));
  p.lds = kRedDoubles * 8 + (size_t(A.ny) * A.f.rs + A.nx + A.ny) * 16;
  return p;
}

template <int MODE>
int launch_fxy(FFTArgs& A, int L, hipStream_t s) {
  PGJ_RUNTIME_FFT(A);
  const PlaneLaunch p = plane_launch(A, L);
  if (int e = allow_lds(fxy_kernel<MODE>, p.lds)) return e;
  hipLaunchKernelGGL(fxy_kernel<MODE>, p.grid, dim3(p.threads), p.lds, s, A);
  PGJ_LAUNCHED("fxy_kernel");
  return PGJ_OK;
}

template <int MODE, int C>
int launch_fz_c(FFTArgs& A, int L, hipStream_t s) {
  const int blocks = (A.ny * A.f.nkx + C - 1) / C;
  PGJ_REQUIRE(A.zslots == blocks && blocks <= A.f.nkb * A.ny, "z pass blocks (%d) do not match the partial layout (%d)",
              blocks, A.zslots);
  const size_t lds = kRedDoubles * 8 + size_t(A.nz) * (3 * C + 1) * 16;
  // a thread per element of the Green multiply, or what the transforms need
  const int threads = std::max(line_threads(A.f.pz, 3 * C), std::min(512, (A.nz * C + 63) / 64 * 64));
  if (int e = allow_lds(fz_kernel<MODE, C>, lds)) return e;
  hipLaunchKernelGGL((fz_kernel<MODE, C>), dim3(blocks, 1, L), dim3(threads), lds, s, A);
  PGJ_LAUNCHED("fz_kernel");
  return PGJ_OK;
}

template <int MODE>
int launch_fz(FFTArgs& A, int L, hipStream_t s) {
  PGJ_RUNTIME_FFT(A);
  switch (A.zkc) {
    case 16: return launch_fz_c<MODE, 16>(A, L, s);
    case 8: return launch_fz_c<MODE, 8>(A, L, s);
    default: return launch_fz_c<MODE, 4>(A, L, s);
  }
}

template <int MODE>
int launch_fxyi(FFTArgs& A, int L, hipStream_t s) {
  PGJ_RUNTIME_FFT(A);
  const PlaneLaunch p = plane_launch(A, L);
  if (int e = allow_lds(fxyi_kernel<MODE>, p.lds)) return e;
  hipLaunchKernelGGL(fxyi_kernel<MODE>, p.grid, dim3(p.threads), p.lds, s, A);
  PGJ_LAUNCHED("fxyi_kernel");
  return PGJ_OK;
}

// 16 columns (two lines of every row) where that still gives a block per CU and the columns stay within 64 KB, 8 down to
// 100 blocks, else 4. Preconditioner with 4 / 8 / 16 columns (us): 20^3 one load 20.3 / 20.9 / 21.9, 40^3 three loads
// 35.5 / 33.1 / 33.5, 45x60x50 one 36.4 / 33.2 / 34.2, three 48.3 / 51.3 / 46.7, 60x50x54 six 97.9 / 94.5 / 89.7,
// 98x35x80 three (73 KB at 16) 107 / 109 / 126.
int runtime_chunk(const FFTGeom& f, int L) {
  const int pl = f.ny * f.nkx;
  int c = 16;
  while (c > kMinChunk &&
         (int64_t(pl + c - 1) / c * L < (c == 16 ? 256 : 100) || size_t(f.nz) * 3 * c * 16 > 64 * 1024))
    c /= 2;
  return c;
}

int launch_fxy_mode(FFTArgs& A, int L, int mode, hipStream_t s) {
  switch (mode) {
    case kFxyScale: return launch_fxy<kFxyScale>(A, L, s);
    case kFxyPre: return launch_fxy<kFxyPre>(A, L, s);
    default: return launch_fxy<kFxyPCG>(A, L, s);
  }
}

int launch_fz_mode(FFTArgs& A, int L, int mode, hipStream_t s) {
  switch (mode) {
    case kFzScale: return launch_fz<kFzScale>(A, L, s);
    case kFzPre: return launch_fz<kFzPre>(A, L, s);
    case kFzInit: return launch_fz<kFzInit>(A, L, s);
    default: return launch_fz<kFzPCG>(A, L, s);
  }
}

int launch_fxyi_mode(FFTArgs& A, int L, int mode, hipStream_t s) {
  return mode == kFxyiPre ? launch_fxyi<kFxyiPre>(A, L, s) : launch_fxyi<kFxyiPCG>(A, L, s);
}

}  // namespace pgj

using namespace pgj;

extern "C" size_t pgj_plan_bytes(const pgj_grid* g) { return plan_layout(*g).bytes; }

extern "C" int pgj_plan_init(const pgj_grid* g, void* plan, void* stream) {
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(plan != nullptr, "null plan");
  PGJ_REQUIRE(g->hx > 0 && g->hy > 0 && g->hz > 0 && g->mu > 0 && g->lam + g->mu > 0, "invalid voxel or medium");
  PlanLayout pl = plan_layout(*g);
  char* b = static_cast<char*>(plan);
  hipStream_t s = as_stream(stream);
  const int nmax = max(g->nx, max(g->ny, g->nz));
  hipLaunchKernelGGL(plan_twiddles, dim3((nmax + 255) / 256), dim3(256), 0, s, g->nx, g->ny, g->nz,
                     reinterpret_cast<double2*>(b + pl.tw_x), reinterpret_cast<double2*>(b + pl.tw_y),
                     reinterpret_cast<double2*>(b + pl.tw_z));
  PGJ_LAUNCHED("plan_twiddles");
  const FFTGeom f = fft_geom(*g);
  hipLaunchKernelGGL(plan_symbol, dim3(unsigned((f.nf + 255) / 256)), dim3(256), 0, s, g->nz, g->ny, g->nx, g->hx,
                     g->hy, g->hz, g->lam, g->mu, reinterpret_cast<double*>(b + pl.sym));
  PGJ_LAUNCHED("plan_symbol");
  return PGJ_OK;
}

extern "C" int pgj_fi_coeff(const pgj_grid* g, double* out4, double* vtab, void* stream) {
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(out4, "null output");
  const FFTGeom f = fft_geom(*g);
  hipLaunchKernelGGL(fi_coeff_kernel, dim3(unsigned((f.nf + 255) / 256)), dim3(256), 0, as_stream(stream), g->nz,
                     g->ny, g->nx, g->hx, g->hy, g->hz, g->lam, g->mu, out4, vtab);
  PGJ_LAUNCHED("fi_coeff_kernel");
  return PGJ_OK;
}

extern "C" int pgj_plan_symbol(const pgj_grid* g, const void* plan, double* out, void* stream) {
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(plan && out, "null plan or output");
  const FFTGeom f = fft_geom(*g);
  PlanLayout pl = plan_layout(*g);
  hipError_t e = hipMemcpyAsync(out, static_cast<const char*>(plan) + pl.sym, size_t(6) * f.nf * 8,
                                hipMemcpyDeviceToDevice, as_stream(stream));
  if (e != hipSuccess) {
    set_error("symbol copy failed: %s", hipGetErrorString(e));
    return PGJ_ERR_HIP;
  }
  return PGJ_OK;
}

extern "C" size_t pgj_precond_ws_bytes(const pgj_grid* g, int L) {
  if (!g) return 0;
  return precond_layout(*g, L).bytes;
}

extern "C" int pgj_scale_spectrum(const pgj_grid* g, const void* plan, const double* s, void* s_hat, void* ws,
                                  void* stream) {
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(plan && s && s_hat && ws, "invalid scale spectrum arguments");
  FFTArgs A = fft_args(*g, plan);
  PrecondLayout pl = precond_layout(*g, 1);
  if (static_fft(*g)) {
    // the compile-time passes read s in its (1, 3N) node-interleaved layout
    A.s = s;
    A.soa = 0;
    A.spec = static_cast<double2*>(s_hat);
    A.pr = reinterpret_cast<double*>(static_cast<char*>(ws) + pl.pr);
    A.pg = reinterpret_cast<double*>(static_cast<char*>(ws) + pl.pg);
    zpass_choose(A, *g, 1);
    hipStream_t st = as_stream(stream);
    if (int e = launch_fxy_static(A, 1, kFxyScale, st)) return e;
    return launch_fz_static(A, 1, kFzScale, st);
  }
  A.s = s;
  A.spec = static_cast<double2*>(s_hat);
  A.pr = reinterpret_cast<double*>(static_cast<char*>(ws) + pl.pr);
  A.pg = reinterpret_cast<double*>(static_cast<char*>(ws) + pl.pg);
  zpass_choose(A, *g, 1);
  hipStream_t st = as_stream(stream);
  if (int e = launch_fxy<kFxyScale>(A, 1, st)) return e;
  return launch_fz<kFzScale>(A, 1, st);
}

namespace pgj {

// z, or with `dir` (L = 1) the fields pdir, rz_old and rz_out of it.
static int precond_passes(const pgj_grid* g, int L, const void* plan, const double* r, const double* s, const void* s_hat,
                          double* z, const FFTArgs* dir, void* ws, hipStream_t st) {
  FFTArgs A = fft_args(*g, plan);
  if (dir) {
    A.pdir = dir->pdir;
    A.rz_old = dir->rz_old;
    A.rz_out = dir->rz_out;
  }
  PrecondLayout pl = precond_layout(*g, L);
  if (static_fft(*g)) {
    // the compile-time passes read r and s and write z in their (L, 3N) node-interleaved layout; r is read by
    // the forward pass only, so z may alias it
    char* w = static_cast<char*>(ws);
    A.rin = r;
    A.s = s;
    A.shat = static_cast<const double2*>(s_hat);
    A.spec = reinterpret_cast<double2*>(w + pl.spec);
    A.pr = reinterpret_cast<double*>(w + pl.pr);
    A.pg = reinterpret_cast<double*>(w + pl.pg);
    A.zout = z;
    A.soa = 0;
    zpass_choose(A, *g, L);
    if (int e = launch_fxy_static(A, L, kFxyPre, st)) return e;
    if (int e = launch_fz_static(A, L, kFzPre, st)) return e;
    return launch_fxyi_static(A, L, st, dir ? kFxyiDir : kFxyiPre);
  }
  char* w = static_cast<char*>(ws);
  A.rin = r;
  A.s = s;
  A.shat = static_cast<const double2*>(s_hat);
  A.spec = reinterpret_cast<double2*>(w + pl.spec);
  A.pr = reinterpret_cast<double*>(w + pl.pr);
  A.pg = reinterpret_cast<double*>(w + pl.pg);
  A.zout = z;
  zpass_choose(A, *g, L);
  if (int e = launch_fxy<kFxyPre>(A, L, st)) return e;
  if (int e = launch_fz<kFzPre>(A, L, st)) return e;
  return dir ? launch_fxyi<kFxyiDir>(A, L, st) : launch_fxyi<kFxyiPre>(A, L, st);
}

int precond_direction(const pgj_grid& g, const void* plan, const double* r, const double* s, const void* s_hat, double* p,
                      const double* rz_old, double* rz, void* ws, hipStream_t stream) {
  FFTArgs dir{};
  dir.pdir = p;
  dir.rz_old = rz_old;
  dir.rz_out = rz;
  return precond_passes(&g, 1, plan, r, s, s_hat, nullptr, &dir, ws, stream);
}

}  // namespace pgj

extern "C" int pgj_precond_apply(const pgj_grid* g, int L, const void* plan, const double* r, const double* s,
                                 const void* s_hat, double* z, void* ws, void* stream) {
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && plan && r && z && ws, "invalid preconditioner arguments");
  PGJ_REQUIRE((s == nullptr) == (s_hat == nullptr), "s and s_hat must be given together");
  return precond_passes(g, L, plan, r, s, s_hat, z, nullptr, ws, as_stream(stream));
}
