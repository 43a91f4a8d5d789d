// Vector kernels of the generic batched PCG (solve_pcg_batched) on (B, n)
// row-major FP64 or FP32 vectors (sums and scalars in FP64): dot-product partials reduced in a fixed order, the
// fused alpha/u/r update with |r|^2 partials, the per-batch relative residual /
// best-iterate / convergence-latch finalization, the fused (optionally Jacobi)
// z / r.z / beta / p update. Semantics follow
// solver/src/runtime/fi/source/femlib/batched/pcg.py:75-245 (eager loop),
// :636-669 (compiled pre/post steps), :677-727 (latch kernels, best copy).
#include <algorithm>
#include <cmath>

#include "fft_kernels.h"
#include "hex8_kernels.h"
#include "layout.h"
#include "pgj_internal.h"

namespace pgj {

constexpr int kVecThreads = 256;
constexpr double kPcgEps = 1e-30;  // pcg.py:112 (eps clamp of pAp and rz)

// Blocks per batch, at most 1024. One value per thread while the launch has at most 2048 blocks (a round of them): a pass
// over a small vector is one round trip to memory, and every further value of a thread would add its own (four values:
// certified solve 32^3 3.17 ms, one: 3.10; generic composite C^H 48^3 16.7 and 16.2 ms). Four values in larger launches,
// because every block of an update reads all partials of its batch, which came to more than its values (pre-step, one
// value against four: 6 x 262144 37 / 24 us, 64 x 98304 114 / 72, 3 x 331776 20.9 / 20.2, and 6 x 98304 17.8 / 18.4).
inline int vec_blocks(int B, int64_t n) {
  const int64_t one = std::min<int64_t>((n + kVecThreads - 1) / kVecThreads, 1024);
  if (B * one <= 2048) return int(one);
  return int(std::min<int64_t>((n + 4 * kVecThreads - 1) / (4 * kVecThreads), 1024));
}

// Batches whose latches the first block of pcg_best forms itself, four reductions at a time; more of them take a launch
// of their own, which costs 2.5 us (256 batches of 3000 values: the pre-step 37 us with the latches in the block, 19).
constexpr int kLatchBatches = 32;

#define PGJ_GRID_LOOP(i, n)                                                                      \
  _Pragma("unroll 4") for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < (n); \
                           i += int64_t(gridDim.x) * blockDim.x)

// r = rhs - Ax (Ax may be null: r = rhs); rhs_part[b][blk] = partial |rhs_b|^2.
// Vectors are T (FP64 or FP32); sums, partials and per-batch scalars are FP64.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_start(const T* rhs, const T* Ax, T* r, int64_t n,
                                                         double* rhs_part) {
  __shared__ double red[kVecThreads / 64];
  const int64_t off = int64_t(blockIdx.y) * n;
  double s = 0.0;
  PGJ_GRID_LOOP(i, n) {
    const T f = rhs[off + i];
    r[off + i] = Ax ? T(f - Ax[off + i]) : f;
    s = fma(double(f), double(f), s);
  }
  const double t = block_sum(s, red);
  if (threadIdx.x == 0) rhs_part[int64_t(blockIdx.y) * gridDim.x + blockIdx.x] = t;
}

// rhs_norm[b] = max(sqrt(sum of partials), 1e-30), one wavefront per batch.
__global__ void pcg_norms(int B, const double* part, int nblk, double* out) {
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int b = blockIdx.x * nw + wave; b < B; b += gridDim.x * nw) {
    const double s = wave_reduce_partials(part + int64_t(b) * nblk, nblk, 1);
    if ((threadIdx.x & 63) == 0) out[b] = fmax(sqrt(s), 1e-30);
  }
}

// part[b][blk] = partial x_b . y_b; with minv, z = minv * x is stored and y is ignored (Jacobi r.z). With `rz`, its
// value goes to `rz_old`, so that the pass after this one can replace rz while its blocks still read the old one.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_dot(const T* x, const T* y, const T* minv, T* z, int64_t n,
                                                       int64_t minv_stride, double* part, const double* rz,
                                                       double* rz_old) {
  __shared__ double red[kVecThreads / 64];
  if (rz && blockIdx.x == 0 && threadIdx.x == 0) rz_old[blockIdx.y] = rz[blockIdx.y];
  const int64_t off = int64_t(blockIdx.y) * n;
  const int64_t moff = int64_t(blockIdx.y) * minv_stride;
  double s = 0.0;
  PGJ_GRID_LOOP(i, n) {
    const T xv = x[off + i];
    T yv;
    if (minv) {
      yv = xv * minv[moff + i];
      z[off + i] = yv;
    } else {
      yv = y[off + i];
    }
    s = fma(double(xv), double(yv), s);
  }
  const double t = block_sum(s, red);
  if (threadIdx.x == 0) part[int64_t(blockIdx.y) * gridDim.x + blockIdx.x] = t;
}

// Per batch: reduce partials to a scalar (one wavefront each).
__global__ void pcg_reduce(int B, const double* part, int nblk, double* out) {
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int b = blockIdx.x * nw + wave; b < B; b += gridDim.x * nw) {
    const double s = wave_reduce_partials(part + int64_t(b) * nblk, nblk, 1);
    if ((threadIdx.x & 63) == 0) out[b] = s;
  }
}

// alpha = rz / max(pAp, eps), 0 where pAp is not finite or <= 0; u += alpha p;
// r -= alpha Ap; rr_part = partial |r|^2 of the updated residual. The best residuals and the stop iteration so far go
// to `best_old` and `stop_old` for pcg_best, whose blocks read them while others already write the new ones; rz goes to
// `rz_old` likewise, for the steps of pgj_pcg_fi_iterate.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_update_ur(T* __restrict__ u, T* __restrict__ r,
                                                             const T* __restrict__ p,
                                                             const T* __restrict__ Ap, int64_t n,
                                                             const double* pap_part, int nblk, const double* rz,
                                                             double* rr_part, const double* best_res,
                                                             const int64_t* state, double* best_old,
                                                             int64_t* stop_old, double* rz_old) {
  __shared__ double red[kVecThreads / 64];
  __shared__ double s_alpha;
  const int b = blockIdx.y;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    best_old[b] = best_res[b];
    rz_old[b] = rz[b];
    if (b == 0) *stop_old = state[0];
  }
  if (threadIdx.x < 64) {
    const double pap = wave_reduce_partials(pap_part + int64_t(b) * nblk, nblk, 1);
    if (threadIdx.x == 0) {
      const bool bad = !isfinite(pap) || pap <= 0.0;
      s_alpha = bad ? 0.0 : rz[b] / fmax(pap, kPcgEps);
    }
  }
  __syncthreads();
  const T alpha = T(s_alpha);
  const int64_t off = int64_t(b) * n;
  double s = 0.0;
  PGJ_GRID_LOOP(i, n) {
    u[off + i] = fma(alpha, p[off + i], u[off + i]);
    const T rn = fma(-alpha, Ap[off + i], r[off + i]);
    r[off + i] = rn;
    s = fma(double(rn), double(rn), s);
  }
  const double t = block_sum(s, red);
  if (threadIdx.x == 0) rr_part[int64_t(b) * gridDim.x + blockIdx.x] = t;
}

// res = sqrt(|r|^2) / rhs_norm; improved = res < best_res (latched: and no stop recorded yet); best_res updated and u
// copied to best_u where improved. Latched: state[0] (stop iteration) is set to `iteration` the first time every
// res < tol; state[1] to 1 the first time every res < near_tol (near_tol > 0 only), by the first block for up to
// kLatchBatches batches, else by pcg_latch. Every block
// forms its batch's residual from the partials (at most 1024, one pass of a wavefront), which costs it less than the
// launch of its own that this test took before the copy: 2.9 of 24 us of vector kernels an iteration at 32^3.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_best(const T* __restrict__ u, T* __restrict__ best_u,
                                                        int64_t n, int B, const double* rr_part,
                                                        int nblk, const double* rhs_norm, const double* best_old,
                                                        const int64_t* stop_old, double* res, double* best_res,
                                                        uint8_t* improved, int64_t* state, double tol, double near_tol,
                                                        int64_t iteration, int latched) {
  const int b = blockIdx.y, wave = threadIdx.x >> 6;
  const int64_t stopped = latched ? *stop_old : 0;
  const double rv = sqrt(wave_reduce_partials(rr_part + int64_t(b) * nblk, nblk, 1)) / rhs_norm[b];
  const bool imp = rv < best_old[b] && stopped == 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    res[b] = rv;
    improved[b] = imp;
    if (imp) best_res[b] = rv;
  }
  if (imp) {
    const int64_t off = int64_t(b) * n;
    PGJ_GRID_LOOP(i, n) best_u[off + i] = u[off + i];
  }
  if (!latched || B > kLatchBatches || blockIdx.x != 0 || b != 0) return;
  int ok = rv < tol, near = rv < near_tol;
  for (int k = 1 + wave; k < B; k += kVecThreads / 64) {
    const double v = sqrt(wave_reduce_partials(rr_part + int64_t(k) * nblk, nblk, 1)) / rhs_norm[k];
    ok &= v < tol;
    near &= v < near_tol;
  }
  const int all_ok = __syncthreads_and(ok);
  const int all_near = __syncthreads_and(near);
  if (threadIdx.x == 0) {
    if (stopped == 0 && all_ok) state[0] = iteration;
    if (near_tol > 0.0 && state[1] == 0 && all_near) state[1] = 1;
  }
}

// The latches of more than kLatchBatches batches from the residuals that pcg_best left. One block.
__global__ __launch_bounds__(1024) void pcg_latch(int B, const double* res, int64_t* state, double tol, double near_tol,
                                                  int64_t iteration) {
  int ok = 1, near = 1;
  for (int b = threadIdx.x; b < B; b += 1024) {
    ok &= res[b] < tol;
    near &= res[b] < near_tol;
  }
  const int all_ok = __syncthreads_and(ok);
  const int all_near = __syncthreads_and(near);
  if (threadIdx.x == 0) {
    if (state[0] == 0 && all_ok) state[0] = iteration;
    if (near_tol > 0.0 && state[1] == 0 && all_near) state[1] = 1;
  }
}

// beta = rz_new / max(rz_old, eps); p = z + beta p; rz = rz_new.
template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_update_p(const T* __restrict__ z, T* __restrict__ p, int64_t n,
                                                            const double* rz_part, int nblk, const double* rz_old,
                                                            double* rz) {
  const int b = blockIdx.y;
  const double rzn = wave_reduce_partials(rz_part + int64_t(b) * nblk, nblk, 1);
  const T beta = T(rzn / fmax(rz_old[b], kPcgEps));
  if (blockIdx.x == 0 && threadIdx.x == 0) rz[b] = rzn;
  const int64_t off = int64_t(b) * n;
  PGJ_GRID_LOOP(i, n) p[off + i] = fma(beta, p[off + i], z[off + i]);
}

template <typename T>
__global__ __launch_bounds__(kVecThreads) void pcg_copy(const T* x, T* y, int64_t total) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += int64_t(gridDim.x) * blockDim.x)
    y[i] = x[i];
}

inline dim3 batch_grid(int B) { return dim3((B + 3) / 4); }

}  // namespace pgj

using namespace pgj;

namespace {
bool pcg_shape_ok(int B, int64_t n) { return B >= 1 && B <= 65535 && n >= 1 && n <= (int64_t(1) << 40); }

// Workspace in doubles: partials of p.Ap, |r|^2 and r.z (B x nblk each), then the values a pass replaces while its blocks
// read them: best residuals (B), r.z (B), stop iteration.
struct PcgWs {
  size_t pap, rr, rz, best_old, rz_old, stop_old, doubles;
};
PcgWs pcg_ws(int B, int64_t n) {
  const size_t row = size_t(B) * vec_blocks(B, n);
  PcgWs w{};
  w.rr = row;
  w.rz = 2 * row;
  w.best_old = 3 * row;
  w.rz_old = w.best_old + B;
  w.stop_old = w.rz_old + B;
  w.doubles = w.stop_old + 1;
  return w;
}
}  // namespace

extern "C" size_t pgj_pcg_ws_bytes(int B, int64_t n) {
  if (!pcg_shape_ok(B, n)) return 0;
  return align256(pcg_ws(B, n).doubles * 8);
}

namespace {
template <typename T>
int pcg_start_t(int B, int64_t n, const T* rhs, const T* Ax, T* r, double* rhs_norm, double* ws, void* stream) {
  PGJ_REQUIRE(pcg_shape_ok(B, n) && rhs && r && rhs_norm && ws, "invalid pcg start arguments");
  hipStream_t s = as_stream(stream);
  const int nblk = vec_blocks(B, n);
  hipLaunchKernelGGL(pcg_start<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, rhs, Ax, r, n, ws);
  PGJ_LAUNCHED("pcg_start");
  hipLaunchKernelGGL(pcg_norms, batch_grid(B), dim3(256), 0, s, B, ws, nblk, rhs_norm);
  PGJ_LAUNCHED("pcg_norms");
  return PGJ_OK;
}

template <typename T>
int pcg_init_t(int B, int64_t n, const T* r, const T* z, T* p, double* rz, double* ws, void* stream) {
  PGJ_REQUIRE(pcg_shape_ok(B, n) && r && z && p && rz && ws, "invalid pcg init arguments");
  hipStream_t s = as_stream(stream);
  const int nblk = vec_blocks(B, n);
  hipLaunchKernelGGL(pcg_dot<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, r, z, nullptr, nullptr, n, int64_t(0), ws,
                     nullptr, nullptr);
  PGJ_LAUNCHED("pcg_dot");
  hipLaunchKernelGGL(pcg_reduce, batch_grid(B), dim3(256), 0, s, B, ws, nblk, rz);
  PGJ_LAUNCHED("pcg_reduce");
  const int64_t total = int64_t(B) * n;
  const int64_t g = (total + kVecThreads * 4 - 1) / (kVecThreads * 4);
  hipLaunchKernelGGL(pcg_copy<T>, dim3(unsigned(g < 4096 ? g : 4096)), dim3(kVecThreads), 0, s, z, p, total);
  PGJ_LAUNCHED("pcg_copy");
  return PGJ_OK;
}

template <typename T>
int pcg_pre_step_t(int B, int64_t n, T* u, T* r, const T* p, const T* Ap, const double* rz, const double* rhs_norm,
                   T* best_u, double* best_res, double* res, uint8_t* improved, int64_t* state, double tol,
                   double near_tol, int64_t iteration, int latched, double* ws, void* stream) {
  PGJ_REQUIRE(pcg_shape_ok(B, n) && u && r && p && Ap && rz && rhs_norm && best_u && best_res && res && improved &&
                  state && ws,
              "invalid pcg pre-step arguments");
  hipStream_t s = as_stream(stream);
  const int nblk = vec_blocks(B, n);
  const PcgWs w = pcg_ws(B, n);
  double *pap = ws + w.pap, *rr = ws + w.rr, *best_old = ws + w.best_old;
  int64_t* stop_old = reinterpret_cast<int64_t*>(ws + w.stop_old);
  hipLaunchKernelGGL(pcg_dot<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, p, Ap, nullptr, nullptr, n, int64_t(0), pap,
                     nullptr, nullptr);
  PGJ_LAUNCHED("pcg_dot");
  hipLaunchKernelGGL(pcg_update_ur<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, u, r, p, Ap, n, pap, nblk, rz, rr,
                     best_res, state, best_old, stop_old, ws + w.rz_old);
  PGJ_LAUNCHED("pcg_update_ur");
  hipLaunchKernelGGL(pcg_best<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, u, best_u, n, B, rr, nblk, rhs_norm, best_old,
                     stop_old, res, best_res, improved, state, tol, near_tol, iteration, latched);
  PGJ_LAUNCHED("pcg_best");
  if (latched && B > kLatchBatches) {
    hipLaunchKernelGGL(pcg_latch, dim3(1), dim3(1024), 0, s, B, res, state, tol, near_tol, iteration);
    PGJ_LAUNCHED("pcg_latch");
  }
  return PGJ_OK;
}

template <typename T>
int pcg_post_step_t(int B, int64_t n, const T* r, T* z, const T* minv, int64_t minv_stride, T* p, double* rz,
                    double* ws, void* stream) {
  PGJ_REQUIRE(pcg_shape_ok(B, n) && r && z && p && rz && ws && (minv_stride == 0 || minv_stride == n),
              "invalid pcg post-step arguments");
  hipStream_t s = as_stream(stream);
  const int nblk = vec_blocks(B, n);
  const PcgWs w = pcg_ws(B, n);
  double *part = ws + w.rz, *rz_old = ws + w.rz_old;
  hipLaunchKernelGGL(pcg_dot<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, r, z, minv, z, n, minv_stride, part, rz,
                     rz_old);
  PGJ_LAUNCHED("pcg_dot");
  hipLaunchKernelGGL(pcg_update_p<T>, dim3(nblk, B), dim3(kVecThreads), 0, s, z, p, n, part, nblk, rz_old, rz);
  PGJ_LAUNCHED("pcg_update_p");
  return PGJ_OK;
}
}  // namespace

extern "C" int pgj_pcg_start(int B, int64_t n, const double* rhs, const double* Ax, double* r, double* rhs_norm,
                             double* ws, void* stream) {
  return pcg_start_t(B, n, rhs, Ax, r, rhs_norm, ws, stream);
}

extern "C" int pgj_pcg_init(int B, int64_t n, const double* r, const double* z, double* p, double* rz, double* ws,
                            void* stream) {
  return pcg_init_t(B, n, r, z, p, rz, ws, stream);
}

extern "C" int pgj_pcg_pre_step(int B, int64_t n, double* u, double* r, const double* p, const double* Ap,
                                const double* rz, const double* rhs_norm, double* best_u, double* best_res,
                                double* res, uint8_t* improved, int64_t* state, double tol, double near_tol,
                                int64_t iteration, int latched, double* ws, void* stream) {
  return pcg_pre_step_t(B, n, u, r, p, Ap, rz, rhs_norm, best_u, best_res, res, improved, state, tol, near_tol,
                        iteration, latched, ws, stream);
}

extern "C" int pgj_pcg_post_step(int B, int64_t n, const double* r, double* z, const double* minv,
                                 int64_t minv_stride, double* p, double* rz, double* ws, void* stream) {
  return pcg_post_step_t(B, n, r, z, minv, minv_stride, p, rz, ws, stream);
}

extern "C" int pgj_pcg32_start(int B, int64_t n, const float* rhs, const float* Ax, float* r, double* rhs_norm,
                               double* ws, void* stream) {
  return pcg_start_t(B, n, rhs, Ax, r, rhs_norm, ws, stream);
}

extern "C" int pgj_pcg32_init(int B, int64_t n, const float* r, const float* z, float* p, double* rz, double* ws,
                              void* stream) {
  return pcg_init_t(B, n, r, z, p, rz, ws, stream);
}

extern "C" int pgj_pcg32_pre_step(int B, int64_t n, float* u, float* r, const float* p, const float* Ap,
                                  const double* rz, const double* rhs_norm, float* best_u, double* best_res,
                                  double* res, uint8_t* improved, int64_t* state, double tol, double near_tol,
                                  int64_t iteration, int latched, double* ws, void* stream) {
  return pcg_pre_step_t(B, n, u, r, p, Ap, rz, rhs_norm, best_u, best_res, res, improved, state, tol, near_tol,
                        iteration, latched, ws, stream);
}

extern "C" int pgj_pcg32_post_step(int B, int64_t n, const float* r, float* z, const float* minv,
                                   int64_t minv_stride, float* p, double* rz, double* ws, void* stream) {
  return pcg_post_step_t(B, n, r, z, minv, minv_stride, p, rz, ws, stream);
}

// One load of the scalar operator with its Green preconditioner: what pgj_precond_apply, pgj_pcg_post_step, pgj_hex8_apply
// and pgj_pcg_pre_step do, `count` times, from one call. p.Ap comes from the apply's own blocks, r.z from the z pass of
// the preconditioner (Parseval), and the inverse pass writes p in place of z: six launches an iteration instead of nine,
// with no host work between them. At 32^3 the loop over four entry points was bound by the host, 73 us an iteration for
// 45 us of kernels; now 43.
extern "C" size_t pgj_pcg_fi_ws_bytes(const pgj_grid* g) {
  return g ? align256(size_t(hex8_blocks_bound(*g)) * 8) : 0;
}

extern "C" int pgj_pcg_fi_iterate(const pgj_grid* g, const double* a, const void* plan, const double* sc,
                                  const void* s_hat, double* u, double* r, double* p, double* Ap, double* rz,
                                  const double* rhs_norm, double* best_u, double* best_res, double* res,
                                  uint8_t* improved, int64_t* state, double tol, double near_tol, int64_t iteration,
                                  int count, int latched, double* ws, double* fi_ws, void* precond_ws, void* stream) {
  if (int e = check_grid(g)) return e;
  if (int e = check_fft(g)) return e;
  PGJ_REQUIRE(a && plan && u && r && p && Ap && rz && rhs_norm && best_u && best_res && res && improved && state &&
                  ws && fi_ws && precond_ws && count >= 0 && (sc == nullptr) == (s_hat == nullptr),
              "invalid pcg iterate arguments");
  hipStream_t s = as_stream(stream);
  const int64_t n = int64_t(g->nx) * g->ny * g->nz * 3;
  const int nblk = vec_blocks(1, n);
  const PcgWs w = pcg_ws(1, n);
  double *rr = ws + w.rr, *best_old = ws + w.best_old, *rz_old = ws + w.rz_old;
  int64_t* stop_old = reinterpret_cast<int64_t*>(ws + w.stop_old);
  const bool march = rowmarch_config(*g, 1).valid;
  for (int k = 0; k < count; ++k) {
    if (int e = precond_direction(*g, plan, r, sc, s_hat, p, rz_old, rz, precond_ws, s)) return e;
    const double* pap = fi_ws;
    int pblk;
    if (march) {
      RowArgs A{};
      A.a = a; A.u = p; A.out = Ap; A.ppq = fi_ws;
      if (int e = launch_rowmarch(*g, 1, kModeApplyDot, A, s)) return e;
      pblk = A.cfg.by * A.cfg.bz;  // of the launch itself: a tuner may set another shape meanwhile
    } else {
      if (int e = pgj_hex8_apply(g, 1, a, p, nullptr, Ap, stream)) return e;
      pap = ws + w.pap;
      pblk = nblk;
      hipLaunchKernelGGL(pcg_dot<double>, dim3(nblk, 1), dim3(kVecThreads), 0, s, p, Ap, nullptr, nullptr, n, int64_t(0),
                         ws + w.pap, nullptr, nullptr);
      PGJ_LAUNCHED("pcg_dot");
    }
    hipLaunchKernelGGL(pcg_update_ur<double>, dim3(nblk, 1), dim3(kVecThreads), 0, s, u, r, p, Ap, n, pap, pblk, rz, rr,
                       best_res, state, best_old, stop_old, rz_old);
    PGJ_LAUNCHED("pcg_update_ur");
    hipLaunchKernelGGL(pcg_best<double>, dim3(nblk, 1), dim3(kVecThreads), 0, s, u, best_u, n, 1, rr, nblk, rhs_norm,
                       best_old, stop_old, res, best_res, improved, state, tol, near_tol, iteration + k, latched);
    PGJ_LAUNCHED("pcg_best");
  }
  return PGJ_OK;
}
