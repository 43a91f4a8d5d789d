// Declarations shared by the FFT/Green kernels and the resident solver.
#pragma once

#include "layout.h"
#include "pgj_internal.h"

namespace pgj {

// ------------------------------------------------------------------ arguments
enum { kFxyScale = 0, kFxyPre = 1, kFxyPCG = 2 };
enum { kFzScale = 0, kFzPre = 1, kFzInit = 2, kFzPCG = 3 };
// kFxyiDir: the preconditioner apply that writes the next direction (FFTArgsT::pdir) in place of z, FP64 only. Its own
// instances: the registers of the direction's loads cost the plain apply 5 % (64^3, one load 35.4 -> 37.1 us).
enum { kFxyiPre = 0, kFxyiPCG = 1, kFxyiDir = 2 };

// Arguments of the FFT/Green kernels; T is the vector precision (FP64 plain
// path, FP32 inner solver of the mixed-precision form). Partial sums and the
// PCG scalars stay FP64 in both.
template <typename T>
struct FFTArgsT {
  using C = cplx<T>;
  int nz, ny, nx;
  int64_t N;
  FFTGeom f;
  const C* twx;
  const C* twy;
  const C* twz;
  const T* sym;
  const T* rin;          // fxy pre: input residual
  T* u;                  // fxy pcg
  T* r;                  // fxy pcg
  const T* p;            // fxyi pcg: direction of this iteration (u += alpha p, p_next = z + beta p)
  const T* q;            // fxy pcg
  const T* s;            // scale (nullable)
  const C* shat;         // spectrum of s (nullable)
  C* spec;               // spectrum buffer (L x 3 x nf)
  T* zout;               // fxyi output: z (preconditioner), or the next PCG direction
  double* pr;            // fxy partials  [l][z][c][2] = (sum r^2, sum r)
  double* pg;            // fz partials   [l][blk][4]  = (v.w, s.w_x, s.w_y, s.w_z)
  const double* ppq;     // hex8 partials [l][blk], ppq_count blocks in rows of ppq_stride
  int ppq_count, ppq_stride;
  StateView st;
  int soa;               // vectors (and s) are SoA (L, 3, N) instead of AoS (L, N, 3)
  int group;             // loads per design (s is (designs, 3N), s_hat (designs, 3, nf)); 0: shared
  int zkc, zslots;       // columns per block of the z pass (0: register-resident cubes) and its partial rows per
                         // load, set by zpass_choose. The form follows the radix plan in force at the launch, so in
                         // the PCG modes of the compile-time cubes the passes that sum the rows take their number
                         // from StateView::zrows, where the z pass that wrote them left it: a plan set between the
                         // two (an eager initialization and a captured iteration) changes speed only
  const double* rin64;   // FP32 preconditioner apply on AoS vectors: FP64 input residual, rounded to T on load
  double* zout64;        // ... and FP64 output z (exact widening of the T result); both null otherwise
  double* pdir;          // FP64 preconditioner apply on AoS vectors: p = z + rz / max(rz_old, 1e-30) p takes the place
  const double* rz_old;  // of z, rz (r.z of the z pass) goes to rz_out; one load, all null otherwise
  double* rz_out;
};
using FFTArgs = FFTArgsT<double>;

// r -> p = M^-1 r + beta p of one load (FFTArgsT::pdir); ws as for pgj_precond_apply.
int precond_direction(const pgj_grid& g, const void* plan, const double* r, const double* s, const void* s_hat, double* p,
                      const double* rz_old, double* rz, void* ws, hipStream_t stream);
FFTArgs fft_args(const pgj_grid& g, const void* plan);
int check_fft(const pgj_grid* g);
int launch_fxy_mode(FFTArgs& A, int L, int mode, hipStream_t s);
int launch_fz_mode(FFTArgs& A, int L, int mode, hipStream_t s);
int launch_fxyi_mode(FFTArgs& A, int L, int mode, hipStream_t s);
// Compile-time-shaped SoA kernels for cubic grids (n in 16, 24, 32, 48, 64, 96, 128).
bool static_fft(const pgj_grid& g);
// Whether the LDS z pass of a solve with L loads in all (its workspace's load count) and elements of es bytes
// takes the wide kx chunks: where these fill the device with more than one round of blocks (64^3 FP64).
bool zpass_wide(const pgj_grid& g, int L, int es);
// Columns per block of the runtime z pass (16, 8 or 4) of a workspace of L loads.
int runtime_chunk(const FFTGeom& f, int L);
// Sets A.zkc and A.zslots for a workspace of L loads (FFTArgsT).
template <typename T> void zpass_choose(FFTArgsT<T>& A, const pgj_grid& g, int L);
template <typename T> int launch_fxy_static(FFTArgsT<T>& A, int L, int mode, hipStream_t s);
template <typename T> int launch_fz_static(FFTArgsT<T>& A, int L, int mode, hipStream_t s);
template <typename T> int launch_fxyi_static(FFTArgsT<T>& A, int L, hipStream_t s, int mode = kFxyiPCG);

}  // namespace pgj
