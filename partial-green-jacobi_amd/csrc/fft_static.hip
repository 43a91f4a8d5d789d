// Compile-time-shaped FFT/Green kernels of the resident solver for cubic
// grids n in {16, 24, 32, 48, 64, 96, 128}. Vectors and the scale s are SoA
// (L, 3, N): one block transforms one component plane, so a plane needs only
// n (n/2+1) complex values of LDS (34 KiB at 64^3) and every index is a
// constant expression. Semantics are those of the runtime kernels in fft.hip.
#include <cmath>

#include "fft_kernels.h"
#include "stockham.h"

namespace pgj {

// Waves per SIMD that the LDS of a block allows (160 KiB per CU, 4 SIMDs),
// capped at 4: the register budget the stream batching is compiled for.
constexpr int lds_occupancy(size_t lds, int threads) {
  const int w = int(size_t(160 * 1024) / lds) * (threads / 64) / 4;
  return w < 1 ? 1 : (w > 4 ? 4 : w);
}

template <int N>
struct Cube {
  static constexpr int M = N / 2;             // complex length of the packed x transform
  static constexpr int NKX = N / 2 + 1;       // half-spectrum width
  static constexpr int RS = NKX;              // LDS row stride (complex)
  static constexpr int PLANE = N * N;         // nodes per z-plane
  static constexpr int64_t NF = int64_t(N) * N * NKX;
  static constexpr int TXY = N >= 96 ? 512 : 256;
  // Partial sums of the other passes are added up by the whole block where there are many of them (128^3: 1040 rows of
  // the z pass per load), else by every wave for itself, which needs no barrier.
  static constexpr bool SHARED_SUMS = N >= 96;
  // LDS bytes for complex values of ES bytes: the data, the twiddle table W_N^j
  // (j < N; the same table serves x, y and z on a cube) and a reduction tail
  // of 4 values x 8 waves
  static constexpr size_t lds_xy(size_t es) { return (size_t(N) * RS + N) * es + 4 * 8 * 8; }
  template <typename R>
  static constexpr int occ_xy() { return lds_occupancy(lds_xy(2 * sizeof(R)), TXY); }
  using Rows = Lines<N, N, 0, RS, 1, false>;          // x transforms (length M) on the N rows
  using Cols = Lines<NKX, NKX, 0, 1, RS, true>;       // y transforms (length N) on the NKX columns
  // vector streams of one z-plane: pairs h = threadIdx.x + i TXY (i < ITER) of
  // consecutive x, in chunks of CH pairs per thread whose loads are issued together
  static constexpr int HALF = PLANE / 2;
  static constexpr int ITER = (HALF + TXY - 1) / TXY;
  static constexpr int CH = ITER <= 8 ? ITER : (ITER % 8 == 0 ? 8 : (ITER + 1) / 2);
  static constexpr bool EXACT = HALF % TXY == 0;
};

// Layout of a load's half spectrum between the passes: the columns kx < N/2 as [c][kz][ky][kx], then the Nyquist
// columns kx = N/2 as [c][kz][ky]. A row of the first part is N/2 complex values, so a chunk of 8 (FP64) or 16 (FP32)
// columns is one aligned 128-byte line that one block of the z pass reads and writes whole. In rows of N/2 + 1 values
// every run straddled lines that its neighbours fetched again (128^3 FP32, three loads: 430 MB fetched for 77 MB of
// spectrum and 51 MB of symbol and scale spectrum).
template <int N>
struct Spec {
  static constexpr int M = N / 2;
  static constexpr int64_t MAIN = int64_t(3) * N * N * M;
};

// z pass of a cube in precision R on KC columns of all three components per block: N/2 / KC chunks per ky row, then
// blocks of the Nyquist column, KC ky values each.
template <int N, typename R, int KC>
struct ZPass {
  static_assert((N / 2) % KC == 0 && N % KC == 0, "chunks cover the columns exactly");
  static constexpr int NCH = N / 2 / KC;
  static constexpr int BLOCKS = NCH * N + N / KC;
  static constexpr int TZ = 3 * N * KC >= 4096 ? 512 : 256;
  // columns in LDS: rows of KC + 1 values and components KC values further apart than their N rows, so that the lines
  // of a transform (a power of two apart otherwise) fall on different banks
  static constexpr int KS = KC + 1, CS = N * KS + KC;
  // columns and the twiddle table; the reduction reuses the column storage once the columns are written back
  static constexpr int COLS = 3 * CS;
  static constexpr size_t lds = (size_t(COLS) + N) * 2 * sizeof(R);
  __host__ __device__ static constexpr int slot(int cz, int k) { return cz * KS + cz / N * KC + k; }
  static constexpr int occ = lds_occupancy(lds, TZ);
  static constexpr int per_cu = occ * 4 / (TZ / 64) > 0 ? occ * 4 / (TZ / 64) : 1;  // resident blocks per CU
  using ZCols = Lines<3 * KC, KC, CS, 1, KS, true>;  // z transforms on (component, column)
};

// Chunk widths of the LDS z pass (fz_static), the best of the widths that divide N/2 on launches of one, three and six
// loads: 96^3 FP64 6 columns 31.7 / 68.6 / 127 us (8: 34.0 / 73.6 / 136, 12: 35.9 / 75.8 / 132), 96^3 FP32 8 columns
// 23.7 / 43 / 73 (6: 25.4 / 46 / 82), 64^3 FP64 4 columns 11.9 / 20.4 / 32.2 (8: 13.6 / 20.5 / 30.7: `wide`, six loads).
template <int N, typename R>
struct ZWidths {
  static constexpr bool d = sizeof(R) == 8;
  static constexpr int def = N <= 64 ? 4 : N == 96 ? (d ? 6 : 8) : d ? 8 : 16;
  static constexpr int wide = N == 64 && d ? 8 : def;
};

// Radix plan of a pass whose plan is not set (pgj_fft_set_plan), and of the passes outside the PCG iteration:
// radix 8 first, one LDS stage less at 32 and 64 and 128. Graph-replayed 3-load launches, radix 4 first against
// radix 8 first, fxy / fxyi: 64^3 FP64 23.2 / 23.6 -> 21.6 / 22.4 us, 48^3 12.3 / 13.1 -> 11.7 / 12.5, 32^3 7.2 / 6.7 ->
// 6.9 / 6.3, 128^3 FP32 72.3 / 101.7 -> 67.8 / 98.4. Radix 4 first stays where it is no slower: 16 (4 x 4 against 8 x 2:
// 4.4 / 4.3 against 4.5 / 4.4).
template <int N>
constexpr int default_plan() {
  return N == 16 ? 0 : 1;
}

template <int N, typename R>
int plan_of(int pass) {
  const int plan = fft_plan(N, int(sizeof(R)), pass);
  return plan == 1 ? 1 : plan == 3 ? 0 : default_plan<N>();
}

// Global -> LDS copy of COUNT values in two phases, so that independent work
// can run while the loads are in flight: load() issues every load of a thread
// (surplus lanes load a clamped, in-bounds index), store() writes the LDS slots.
// map(e) is the global index of LDS slot e.
template <int COUNT, int T, typename X>
struct StageIn {
  static constexpr int PER = (COUNT + T - 1) / T;
  X v[PER];
  template <typename Map>
  __device__ inline void load(const X* __restrict__ src, Map map) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = COUNT % T == 0 ? int(threadIdx.x) + k * T : min(int(threadIdx.x) + k * T, COUNT - 1);
      v[k] = src[map(e)];
    }
  }
  template <typename Slot>
  __device__ inline void store(X* lds, Slot slot) const {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = int(threadIdx.x) + k * T;
      if (COUNT % T == 0 || e < COUNT) lds[slot(e)] = v[k];
    }
  }
  __device__ inline void store(X* lds) const {
    store(lds, [](int e) { return e; });
  }
};

// Pair index of chunk slot i of a vector stream, clamped in bounds for loads.
template <int N>
__device__ inline int pair_of(int i) {
  using C = Cube<N>;
  const int h = int(threadIdx.x) + i * C::TXY;
  return C::EXACT ? h : min(h, C::HALF - 1);
}

// ------------------------------------------------------------ forward xy
template <int N, int MODE, typename R, int PLAN = 0>
__global__ __launch_bounds__(Cube<N>::TXY) __attribute__((amdgpu_waves_per_eu(Cube<N>::template occ_xy<R>())))
void fxy_static(FFTArgsT<R> A) {
  using C = Cube<N>;
  using X = cplx<R>;
  constexpr int T = C::TXY;
  extern __shared__ __align__(16) unsigned char smem[];
  X* plane = reinterpret_cast<X*>(smem);
  X* tw = plane + N * C::RS;
  double* red = reinterpret_cast<double*>(tw + N);
  const int z = blockIdx.x, c = blockIdx.y, l = blockIdx.z;
  const int64_t NN = int64_t(N) * N * N;
  if (MODE == kFxyPCG && !A.st.active[l]) return;
  const int64_t off = (int64_t(l) * 3 + c) * NN + int64_t(z) * C::PLANE;
  const int64_t soff = (int64_t(design_of(l, A.group)) * 3 + c) * NN + int64_t(z) * C::PLANE;
  double sq = 0.0, sm = 0.0;
  // two nodes (x even, x+1) per pair: one packed complex of the x transform
  const X* __restrict__ sp = reinterpret_cast<const X*>(A.s + soff);
  const X* __restrict__ rinp = reinterpret_cast<const X*>(A.rin + off);
  X* __restrict__ rp = reinterpret_cast<X*>(A.r + off);
  const X* __restrict__ qp = reinterpret_cast<const X*>(A.q + off);
  const bool scaled = A.s != nullptr;
  // the scale and preconditioner passes also read the drop-in layout (A.soa == 0): xyz triples per node, so
  // component c of the pair's two nodes sits 24 bytes apart (the other components' blocks share the lines in L2)
  const bool aos = MODE != kFxyPCG && !A.soa;
  const int64_t aoff = int64_t(z) * C::PLANE * 3 + c;
  const R* __restrict__ s_aos = aos && scaled ? A.s + int64_t(design_of(l, A.group)) * 3 * NN + aoff : nullptr;
  const R* __restrict__ r_aos = aos && MODE == kFxyPre && A.rin ? A.rin + int64_t(l) * 3 * NN + aoff : nullptr;
  // FP32 apply of FP64 vectors: the residual is read in FP64 and rounded to R
  const bool wide_in = sizeof(R) == 4 && aos && MODE == kFxyPre && A.rin64 != nullptr;
  const double* __restrict__ r64 = wide_in ? A.rin64 + int64_t(l) * 3 * NN + aoff : nullptr;
  auto pair_aos = [](const R* base, int h) {
    const R* q = base + 6 * int64_t(h);
    return c2(q[0], q[3]);
  };
  // rows of z partials to sum: as many as the pass that wrote them left, whatever form a pass launched now would take
  const int zrows = MODE == kFxyPCG ? A.st.zrows[l] : 0;
  double alpha = 0.0;
#pragma unroll
  for (int i0 = 0; i0 < C::ITER; i0 += C::CH) {
    // every load of the chunk is issued before the first use
    X va[C::CH], vb[C::CH], vs[C::CH];
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      const int h = pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1);
      if (MODE == kFxyScale) {
        va[i] = aos ? pair_aos(s_aos, h) : sp[h];
      } else if (MODE == kFxyPre) {
        if (wide_in) {
          const double* q = r64 + 6 * int64_t(h);
          va[i] = c2(R(q[0]), R(q[3]));
        } else {
          va[i] = aos ? pair_aos(r_aos, h) : rinp[h];
        }
      } else {
        va[i] = rp[h];
        vb[i] = qp[h];
      }
      vs[i] = c2(R(1), R(1));
    }
    StageIn<N, T, X> twl;  // the twiddle table, staged with the first chunk
    if (i0 == 0) twl.load(A.twx, [](int e) { return e; });
    // PCG: the step length is reduced while the r and q loads are in flight
    if (MODE == kFxyPCG && i0 == 0) {
      double pq, rz;
      // per-load partials are laid out with the geometry's chunk count (slices of a set are offset by it)
      const double* ppq = A.ppq + int64_t(l) * A.ppq_stride;
      const double* pg = A.pg + int64_t(l) * A.f.nkb * N * 4;
      if (C::SHARED_SUMS) {
        double t[2] = {0.0, 0.0};
        for (int k = threadIdx.x; k < A.ppq_count; k += T) t[0] += ppq[k];
        for (int k = threadIdx.x; k < zrows; k += T) t[1] += pg[4 * k];
        block_sums<2>(t, red);
        pq = t[0];
        rz = t[1];
      } else {
        wave_reduce_partials_2(ppq, A.ppq_count, 1, pg, zrows, 4, pq, rz);
      }
      const bool valid = isfinite(pq) && pq > 0.0 && isfinite(rz) && rz > 0.0;
      alpha = valid ? rz / pq : 0.0;
      if (threadIdx.x == 0 && z == 0 && c == 0) {
        A.st.rz[l] = rz;
        A.st.alpha[l] = alpha;
        A.st.valid[l] = valid;
        A.st.first[l] = 0;
      }
    }
    if (i0 == 0) twl.store(tw);
    if (MODE != kFxyScale && scaled) {
#pragma unroll
      for (int i = 0; i < C::CH; ++i) {
        const int h = pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1);
        vs[i] = aos ? pair_aos(s_aos, h) : sp[h];
      }
    }
    const R ra = R(alpha);
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      const int h = int(threadIdx.x) + (i0 + i) * T;
      if (i0 + i >= C::ITER || (!C::EXACT && h >= C::HALF)) continue;
      X v = va[i];
      if (MODE != kFxyScale) {
        X rn = va[i];
        if (MODE == kFxyPCG) {
          rn = c2(fma(-ra, vb[i].x, va[i].x), fma(-ra, vb[i].y, va[i].y));
          rp[h] = rn;
        }
        sq = fma(double(rn.x), double(rn.x), fma(double(rn.y), double(rn.y), sq));
        sm += double(rn.x) + double(rn.y);
        v = c2(vs[i].x * rn.x, vs[i].y * rn.y);
      }
      const int e = 2 * h;
      const int x = e % N, y = e / N;
      plane[y * C::RS + x / 2] = v;
    }
  }
  if (MODE != kFxyScale) {
    double t[2] = {sq, sm};
    block_sums<2>(t, red);
    if (threadIdx.x == 0) {
      double* p = A.pr + ((int64_t(l) * N + z) * 3 + c) * 2;
      p[0] = t[0];
      p[1] = t[1];
    }
  }
  __syncthreads();
  sfft<false, C::M, typename C::Rows, T, PLAN>(plane, tw, 2);
  // split the packed spectrum of every row into its half spectrum
  constexpr int HALF = C::M / 2, PAIRS = N * (HALF + 1);
  for (int b = threadIdx.x; b < PAIRS; b += T) {
    const int row = b / (HALF + 1), k = b % (HALF + 1);
    X* L = plane + row * C::RS;
    const X zk = L[k % C::M], zm = L[(C::M - k) % C::M];
    const X E = c2(R(0.5) * (zk.x + zm.x), R(0.5) * (zk.y - zm.y));
    const X O = c2(R(0.5) * (zk.y + zm.y), R(-0.5) * (zk.x - zm.x));
    const X wo = cmul(tw[k], O);
    L[k] = cadd(E, wo);
    if (C::M - k != k) L[C::M - k] = conjd(csub(E, wo));
  }
  __syncthreads();
  sfft<false, N, typename C::Cols, T, PLAN>(plane, tw, 1);
  if (MODE == kFxyScale) {
    // the caller's s_hat: rows of N/2 + 1 values
    X* out = A.spec + ((int64_t(l) * 3 + c) * N + z) * int64_t(N) * C::NKX;
    for (int e = threadIdx.x; e < N * C::NKX; e += T) out[e] = plane[e];
  } else {
    X* out = A.spec + int64_t(l) * 3 * C::NF;
    X* row = out + (int64_t(c) * N + z) * (N * C::M);
    for (int e = threadIdx.x; e < N * C::M; e += T) row[e] = plane[e / C::M * C::RS + e % C::M];
    X* nyq = out + Spec<N>::MAIN + (int64_t(c) * N + z) * N;
    for (int y = threadIdx.x; y < N; y += T) nyq[y] = plane[y * C::RS + C::M];
  }
}

// ---------------------------------------------------------------- z + Green
template <int N, int MODE, typename R, int KC, int PLAN = 0>
__global__ __launch_bounds__((ZPass<N, R, KC>::TZ)) __attribute__((amdgpu_waves_per_eu((ZPass<N, R, KC>::occ))))
void fz_static(FFTArgsT<R> A) {
  using C = Cube<N>;
  using X = cplx<R>;
  using Z = ZPass<N, R, KC>;
  constexpr int T = Z::TZ, NKX = C::NKX;
  extern __shared__ __align__(16) unsigned char smem[];
  X* cols = reinterpret_cast<X*>(smem);
  X* tw = cols + Z::COLS;
  double* red = reinterpret_cast<double*>(cols);  // used only after the columns are written back
  // ky is the fastest index: the kx chunks of one ky row (which share lines of the symbol and s_hat) get block ids N
  // apart, a multiple of 8 for every supported N, and so run on the same XCD / L2.
  const int blk = blockIdx.x, l = blockIdx.z;
  const bool nyq = blk >= Z::NCH * N;                       // blocks of the Nyquist column
  const int y = nyq ? (blk - Z::NCH * N) * KC : blk % N;    // ky of column 0
  const int kx0 = nyq ? N / 2 : blk / N * KC;               // kx of column 0
  const bool lead = threadIdx.x == 0 && blk == 0;
  const int64_t NN = int64_t(N) * N * N;
  // the spectrum columns are loaded first (for every load that may continue)
  // and stay in flight through the convergence test and the mean reduction
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
  // the spectrum columns and the twiddle table go to LDS first; they are read after the test below
  // frequency (cz, column) in the rows of N/2 + 1 values of the symbol and s_hat, and in the spectrum (the scale pass
  // transforms s_hat in place)
  const int fcol = nyq ? NKX : 1;
  const int f0 = y * NKX + kx0;
  const bool packed = MODE != kFzScale;
  const int scol = packed ? 1 : fcol;
  const int sstep = !packed ? N * NKX : nyq ? N : N * (N / 2);
  X* S = A.spec + int64_t(l) * 3 * C::NF + (!packed ? int64_t(f0) : nyq ? Spec<N>::MAIN + y : int64_t(y) * (N / 2) + kx0);
  {
    StageIn<3 * N * KC, T, X> in;
    in.load(S, [&](int e) { return e / KC * sstep + e % KC * scol; });
    StageIn<N, T, X> twl;
    twl.load(A.twz, [](int e) { return e; });
    in.store(cols, [](int e) { return Z::slot(e / KC, e % KC); });
    twl.store(tw);
  }
  double mean[3] = {0.0, 0.0, 0.0};
  if (MODE == kFzInit || MODE == kFzPCG) {
    const int lane = threadIdx.x & 63;
    // one pass over the per-plane partials (|r|^2 and the component sums of r)
    double v = 0.0, vm[3] = {0.0, 0.0, 0.0};
    for (int i = lane; i < N; i += 64) {
      const double* p = A.pr + (int64_t(l) * N + i) * 6;
      v += (p[0] + p[2]) + p[4];
      vm[0] += p[1];
      vm[1] += p[3];
      vm[2] += p[5];
    }
    const double res2 = wave_sum(v);
    if (A.shat)
      for (int c = 0; c < 3; ++c) mean[c] = wave_sum(vm[c]) / double(NN);
    bool act;
    if (MODE == kFzInit) {
      act = res2 > A.st.target2[l] && A.st.it[l] < A.st.cap[l] && !A.st.bad[l];
      if (lead) {
        A.st.active_next[l] = act;
        A.st.it_next[l] = A.st.it[l];
        A.st.bad_next[l] = A.st.bad[l];
        A.st.first[l] = 1;
        A.st.stopped[l] = 0;
        A.st.zrows[l] = Z::BLOCKS;
      }
    } else {
      const bool active = A.st.active[l] != 0;
      const bool valid = A.st.valid[l] != 0;  // set by the forward pass of this iteration
      const bool finite = isfinite(res2);
      const int64_t it = A.st.it[l] + (active ? 1 : 0);
      act = active && valid && finite && res2 > A.st.target2[l] && it < A.st.cap[l];
      if (lead) {
        A.st.active_next[l] = act;
        A.st.it_next[l] = it;
        A.st.bad_next[l] = A.st.bad[l] || (active && !valid) || (active && !finite);
        A.st.stopped[l] = active && !act;
        A.st.zrows[l] = Z::BLOCKS;
      }
    }
    if (!act) return;
  } else if (MODE != kFzScale && A.shat) {
    for (int c = 0; c < 3; ++c)
      mean[c] = wave_reduce_partials(A.pr + (int64_t(l) * N * 3 + c) * 2 + 1, N, 6) / double(NN);
  }
  // a fixed number of frequency slots per thread, in groups of GS slots whose
  // symbol and s_hat loads are all issued before the first is used. Where one
  // group of them fits 64 registers it holds every slot and is issued before the
  // forward transform, so the loads stay in flight while it runs.
  constexpr int EPT = (N * KC + T - 1) / T;
  constexpr bool EARLY = EPT * sizeof(R) <= 16;
  constexpr int GS = (EARLY || EPT <= 3) ? EPT : 2;
  constexpr bool FULL = (N * KC) % T == 0;
  const X* __restrict__ shat_d = A.shat ? A.shat + int64_t(design_of(l, A.group)) * 3 * C::NF + f0 : nullptr;
  const R* __restrict__ sym = A.sym + f0;
  auto slot = [&](int k) { return FULL ? int(threadIdx.x) + k * T : min(int(threadIdx.x) + k * T, N * KC - 1); };
  auto freq = [&](int e) { return e / KC * (N * NKX) + e % KC * fcol; };
  R g[GS][6];
  X sh[GS][3];
  auto load_group = [&](int k0) {
#pragma unroll
    for (int i = 0; i < GS; ++i) {
      const int fidx = freq(slot(k0 + i < EPT ? k0 + i : EPT - 1));
#pragma unroll
      for (int j = 0; j < 6; ++j) g[i][j] = sym[j * C::NF + fidx];
#pragma unroll
      for (int c = 0; c < 3; ++c) sh[i][c] = c2(R(0), R(0));
    }
    if (shat_d) {
#pragma unroll
      for (int i = 0; i < GS; ++i) {
        const int fidx = freq(slot(k0 + i < EPT ? k0 + i : EPT - 1));
#pragma unroll
        for (int c = 0; c < 3; ++c) sh[i][c] = shat_d[int64_t(c) * C::NF + fidx];
      }
    }
  };
  if (MODE != kFzScale && EARLY) load_group(0);
  __syncthreads();
  sfft<false, N, typename Z::ZCols, T, PLAN>(cols, tw, 1);
  if (MODE == kFzScale) {
    for (int e = threadIdx.x; e < 3 * N * KC; e += T) S[e / KC * sstep + e % KC * scol] = cols[Z::slot(e / KC, e % KC)];
    return;
  }
  double rz = 0.0, sw[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k0 = 0; k0 < EPT; k0 += GS) {
    if (!(EARLY && k0 == 0)) load_group(k0);
#pragma unroll
    for (int i = 0; i < GS; ++i) {
      const int k = k0 + i;
      const int e = threadIdx.x + k * T;
      if (k >= EPT || (!FULL && e >= N * KC)) continue;
      const int kcol = e % KC, zz = e / KC;
      X v[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c] = cols[Z::slot(c * N + zz, kcol)];
      if (shat_d) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const R mc = R(mean[c]);
          v[c] = c2(fma(-mc, sh[i][c].x, v[c].x), fma(-mc, sh[i][c].y, v[c].y));
        }
      }
      const R g0 = g[i][0], g1 = g[i][1], g2 = g[i][2], g3 = g[i][3], g4 = g[i][4], g5 = g[i][5];
      X w[3];
      w[0] = c2(g0 * v[0].x + g3 * v[1].x + g4 * v[2].x, g0 * v[0].y + g3 * v[1].y + g4 * v[2].y);
      w[1] = c2(g3 * v[0].x + g1 * v[1].x + g5 * v[2].x, g3 * v[0].y + g1 * v[1].y + g5 * v[2].y);
      w[2] = c2(g4 * v[0].x + g5 * v[1].x + g2 * v[2].x, g4 * v[0].y + g5 * v[1].y + g2 * v[2].y);
      const double wgt = (nyq || kx0 + kcol == 0) ? 1.0 : 2.0;
      double t = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) t += double(v[c].x) * double(w[c].x) + double(v[c].y) * double(w[c].y);
      rz = fma(wgt, t, rz);
      if (shat_d) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          sw[c] = fma(wgt, double(sh[i][c].x) * double(w[c].x) + double(sh[i][c].y) * double(w[c].y), sw[c]);
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) cols[Z::slot(c * N + zz, kcol)] = w[c];
    }
  }
  __syncthreads();
  sfft<true, N, typename Z::ZCols, T, PLAN>(cols, tw, 1);
  for (int e = threadIdx.x; e < 3 * N * KC; e += T) S[e / KC * sstep + e % KC * scol] = cols[Z::slot(e / KC, e % KC)];
  double t[4] = {rz, sw[0], sw[1], sw[2]};
  block_sums<4>(t, red);
  if (threadIdx.x == 0) {
    // per-load partials are laid out with the geometry's chunk count (slices of a set are offset by it)
    double* pg = A.pg + (int64_t(l) * A.f.nkb * N + blk) * 4;
    pg[0] = t[0];
    pg[1] = t[1];
    pg[2] = t[2];
    pg[3] = t[3];
  }
}

// ------------------------------------------------------------- z + Green, in registers
// The z pass of a cube n = 8 P with its transforms in registers and no barrier between its phases. A wave holds 8
// columns of one ky row (the Nyquist blocks: 8 ky of kx = n/2), all three components; lane (col, j) the points
// kz = j + 8 r (r < P) of its column. With k = P a + b,
//   X[P a + b] = sum_j W_8^(j a) [ W_n^(j b) sum_r W_P^(r b) x[j + 8 r] ]:
// a P-point transform in the lane, a twiddle, one exchange among the 8 lanes of the column through LDS, and 8-point
// transforms for b = j + 8 q that leave the lane every component of its frequencies, so the Green multiply needs no
// exchange either (where P is no multiple of 8 the last group leaves lanes idle); the inverse mirrors it. LDS carries
// each point four times instead of the 16 of the staged pass (fz_static), and a wave's 24 (64^3) or 48 loads are all in
// flight at once. Bound by memory from three loads on: 128^3 FP64, three loads, 140 us for 450 MB of spectrum, symbol
// and scale spectrum; by its own chain of loads, exchanges and stores on fewer (zkc_of has the times on both sides).

// Cubes whose columns divide into whole waves of the register-resident z pass.
template <int N>
constexpr bool zreg() { return N % 16 == 0; }

template <int N>
struct ZReg {
  static constexpr int P = N / 8, Q = (P + 7) / 8;
  static constexpr int BS = 8 * 8 + 8;      // row of one b: [j][col], padded by half the banks
  template <typename R>
  static constexpr size_t lds() { return size_t(8 * Q) * BS * 2 * sizeof(R); }
  // Blocks of one wave: blocks of four with one row of partials each measured slower (128^3 FP32, three loads: 104 us
  // against 78 us), their 260 blocks per load leave CUs one block longer than others.
  static constexpr int BLOCKS = N / 16 * N + N / 8;
};

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int N, int MODE, typename R, int EU, bool SCALED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(EU))) void fz_reg(FFTArgsT<R> A) {
  using X = cplx<R>;
  using Z = ZReg<N>;
  constexpr int P = Z::P, NKX = N / 2 + 1, Q = Z::Q;
  constexpr bool ALL = P % 8 == 0;   // else the last group of frequencies b = j + 8 q leaves lanes with b >= P idle
  constexpr int64_t NF = int64_t(N) * N * NKX;
  extern __shared__ __align__(16) unsigned char smem[];
  X* buf = reinterpret_cast<X*>(smem);
  const int lane = threadIdx.x, col = lane & 7, j = lane >> 3;
  const int blk = blockIdx.x, l = blockIdx.z;
  const bool nyq = blk >= N / 16 * N;
  const int y = nyq ? (blk - N / 16 * N) * 8 : blk % N;     // ky of column 0
  const int kx0 = nyq ? N / 2 : blk / N * 8;                // kx of column 0
  const bool lead = lane == 0 && blk == 0;
  const int64_t NN = int64_t(N) * N * N;
  if (MODE == kFzPCG && !A.st.active[l]) {
    if (lead) {
      A.st.active_next[l] = 0;
      A.st.it_next[l] = A.st.it[l];
      A.st.bad_next[l] = A.st.bad[l];
      A.st.stopped[l] = 0;
    }
    return;
  }
  // frequency (kz, column) in the rows of N/2 + 1 values of the symbol and s_hat, and in the spectrum (the scale pass
  // transforms s_hat in place)
  const int fcol = nyq ? NKX : 1;
  const bool packed = MODE != kFzScale;
  const int sstep = !packed ? N * NKX : nyq ? N : N * (N / 2);
  // uniform base and row offsets, one 32-bit offset per lane
  X* S = A.spec + int64_t(l) * 3 * NF +
         (!packed ? int64_t(y * NKX + kx0) : nyq ? Spec<N>::MAIN + y : int64_t(y) * (N / 2) + kx0);
  const unsigned so = unsigned(j * sstep + col * (packed ? 1 : fcol));
  int bq[Q];   // b of the lane's groups, in range also for the idle lanes
  bool on[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    on[q] = ALL || j + 8 * q < P;
    bq[q] = on[q] ? j + 8 * q : P - 1;
  }
  unsigned fo[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) fo[q] = unsigned(bq[q] * (N * NKX) + col * fcol);
  X v[3][P > 8 * Q ? P : 8 * Q];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int r = 0; r < P; ++r) v[c][r] = (S + (c * N + 8 * r) * sstep)[so];
  __builtin_amdgcn_sched_barrier(0);
  X tw[P];   // W_n^(j b)
#pragma unroll
  for (int b = 1; b < P; ++b) tw[b] = A.twz[j * b];
  __builtin_amdgcn_sched_barrier(0);
  double mean[3] = {0.0, 0.0, 0.0};
  if (MODE != kFzScale) {
    double ss = 0.0, vm[3] = {0.0, 0.0, 0.0};
    for (int i = lane; i < N; i += 64) {
      const double* p = A.pr + (int64_t(l) * N + i) * 6;
      ss += (p[0] + p[2]) + p[4];
      vm[0] += p[1];
      vm[1] += p[3];
      vm[2] += p[5];
    }
    if (SCALED)
      for (int c = 0; c < 3; ++c) mean[c] = wave_sum(vm[c]) / double(NN);
    if (MODE != kFzPre) {
      const double res2 = wave_sum(ss);
      const int64_t it0 = A.st.it[l];
      const bool bad = A.st.bad[l] != 0;
      // the initialization's test, or the iteration's (the active mask was tested above; `valid` was set by the forward
      // pass of this iteration)
      const bool valid = MODE == kFzInit || A.st.valid[l] != 0, finite = isfinite(res2);
      const int64_t it = it0 + (MODE == kFzPCG ? 1 : 0);
      const bool act = valid && res2 > A.st.target2[l] && it < A.st.cap[l] && (MODE == kFzInit ? !bad : finite);
      if (lead) {
        A.st.active_next[l] = act;
        A.st.it_next[l] = it;
        A.st.bad_next[l] = bad || (MODE == kFzPCG && !(valid && finite));
        A.st.stopped[l] = MODE == kFzPCG && !act;
        if (MODE == kFzInit) A.st.first[l] = 1;
        A.st.zrows[l] = Z::BLOCKS;
      }
      if (!act) return;
    }
  }
  // symbol and s_hat of the lane's frequencies, fetched GS at a time: the first group before the transforms, each later
  // one before the group in hand is used (when needed where P > 8 leaves no registers for that). The scheduling
  // barriers keep it so: moved further up the loads would take the registers of the transforms, further down nothing
  // would cover them.
  constexpr int GS = 2;
  const X* __restrict__ shat_d = SCALED ? A.shat + int64_t(design_of(l, A.group)) * 3 * NF + y * NKX + kx0 : nullptr;
  const R* __restrict__ sym = A.sym + y * NKX + kx0;
  R g[2][GS][6];
  X sh[2][GS][3];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < GS; ++i) {
      const int k = k0 + i, f = P * (k & 7) * (N * NKX);
#pragma unroll
      for (int m = 0; m < 6; ++m) g[k0 / GS & 1][i][m] = (sym + (m * NF + f))[fo[k >> 3]];
      if (SCALED) {
#pragma unroll
        for (int c = 0; c < 3; ++c) sh[k0 / GS & 1][i][c] = (shat_d + (c * NF + f))[fo[k >> 3]];
      }
    }
  };
  constexpr bool AHEAD = P <= 8;
  __builtin_amdgcn_sched_barrier(0);
  if (MODE != kFzScale && AHEAD) fetch(0);
  const X* none = nullptr;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    __builtin_amdgcn_sched_barrier(0);
    X u[P];
#pragma unroll
    for (int r = 0; r < P; ++r) u[r] = v[c][r];
    dft<P, false>(u, none, N, 1);
#pragma unroll
    for (int b = 0; b < P; ++b) buf[b * Z::BS + j * 8 + col] = b == 0 ? u[0] : cmul(u[b], tw[b]);
    wave_lds_fence();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      X w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = buf[bq[q] * Z::BS + i * 8 + col];
      dft<8, false>(w, none, N, 1);
#pragma unroll
      for (int a = 0; a < 8; ++a) v[c][8 * q + a] = w[a];   // frequency kz = P a + b
    }
    wave_lds_fence();
  }
  if (MODE == kFzScale) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        if (on[q]) {
#pragma unroll
          for (int a = 0; a < 8; ++a)
            (S + (c * N + P * a) * sstep)[unsigned(bq[q] * sstep + col * (packed ? 1 : fcol))] = v[c][8 * q + a];
        }
    return;
  }
  const double wgt = (nyq || kx0 + col == 0) ? 1.0 : 2.0;
  double rz = 0.0, sw[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k0 = 0; k0 < 8 * Q; k0 += GS) {
    __builtin_amdgcn_sched_barrier(0);
    if (!AHEAD) fetch(k0);
    else if (k0 + GS < 8 * Q) fetch(k0 + GS);
    const int bf = k0 / GS & 1;
#pragma unroll
    for (int i = 0; i < GS; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      X x[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const R mc = R(mean[c]);
        x[c] = v[c][k0 + i];
        if (SCALED) x[c] = c2(fma(-mc, sh[bf][i][c].x, x[c].x), fma(-mc, sh[bf][i][c].y, x[c].y));
      }
      const R g0 = g[bf][i][0], g1 = g[bf][i][1], g2 = g[bf][i][2], g3 = g[bf][i][3], g4 = g[bf][i][4],
              g5 = g[bf][i][5];
      X w[3];
      w[0] = c2(g0 * x[0].x + g3 * x[1].x + g4 * x[2].x, g0 * x[0].y + g3 * x[1].y + g4 * x[2].y);
      w[1] = c2(g3 * x[0].x + g1 * x[1].x + g5 * x[2].x, g3 * x[0].y + g1 * x[1].y + g5 * x[2].y);
      w[2] = c2(g4 * x[0].x + g5 * x[1].x + g2 * x[2].x, g4 * x[0].y + g5 * x[1].y + g2 * x[2].y);
      double t = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) t += double(x[c].x) * double(w[c].x) + double(x[c].y) * double(w[c].y);
      const double wk = on[(k0 + i) >> 3] ? wgt : 0.0;
      rz = fma(wk, t, rz);
      if (SCALED) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
          sw[c] = fma(wk, double(sh[bf][i][c].x) * double(w[c].x) + double(sh[bf][i][c].y) * double(w[c].y), sw[c]);
      }
#pragma unroll
      for (int c = 0; c < 3; ++c) v[c][k0 + i] = w[c];
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // the twiddles are read again and the rows' offsets formed again (an opaque copy of what they derive from): held
  // through the multiply they would cost its registers
  const X* twz = A.twz;
  unsigned so2 = so;
  asm volatile("" : "+s"(twz), "+v"(so2));
#pragma unroll
  for (int b = 1; b < P; ++b) tw[b] = twz[j * b];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      X w[8];
#pragma unroll
      for (int a = 0; a < 8; ++a) w[a] = v[c][8 * q + a];
      dft<8, true>(w, none, N, 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) buf[(j + 8 * q) * Z::BS + i * 8 + col] = w[i];   // rows b >= P are not read
    }
    wave_lds_fence();
    X u[P];
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const X x = buf[b * Z::BS + j * 8 + col];
      u[b] = b == 0 ? x : cmul(x, conjd(tw[b]));
    }
    wave_lds_fence();
    dft<P, true>(u, none, N, 1);
#pragma unroll
    for (int r = 0; r < P; ++r) (S + (c * N + 8 * r) * sstep)[so2] = u[r];
  }
  rz = wave_sum(rz);
#pragma unroll
  for (int c = 0; c < 3; ++c) sw[c] = wave_sum(sw[c]);
  if (lane == 0) {
    // per-load partials are laid out with the geometry's chunk count (slices of a set are offset by it)
    double* pg = A.pg + (int64_t(l) * A.f.nkb * N + blk) * 4;
    pg[0] = rz;
    for (int c = 0; c < 3; ++c) pg[1 + c] = sw[c];
  }
}

// --------------------------------------------------------------- inverse xy
// MODE kFxyiPre: the preconditioner apply alone (z = P(s w), no PCG state); kFxyiDir: p = z + beta p in its place.
template <int N, int MODE, typename R, int PLAN = 0>
__global__ __launch_bounds__(Cube<N>::TXY) __attribute__((amdgpu_waves_per_eu(Cube<N>::template occ_xy<R>())))
void fxyi_static(FFTArgsT<R> A) {
  using C = Cube<N>;
  using X = cplx<R>;
  constexpr int T = C::TXY;
  constexpr bool PCG = MODE == kFxyiPCG;
  extern __shared__ __align__(16) unsigned char smem[];
  X* plane = reinterpret_cast<X*>(smem);
  X* tw = plane + N * C::RS;
  const int z = blockIdx.x, c = blockIdx.y, l = blockIdx.z;
  const int64_t NN = int64_t(N) * N * N;
  if (PCG && threadIdx.x == 0 && z == 0 && c == 0) {
    A.st.active[l] = A.st.active_next[l];
    A.st.it[l] = A.st.it_next[l];
    A.st.bad[l] = A.st.bad_next[l];
  }
  const int64_t off = (int64_t(l) * 3 + c) * NN + int64_t(z) * C::PLANE;
  // PCG: the displacement update u += alpha p of this iteration (alpha from the forward pass)
  const bool move = PCG && A.p != nullptr && A.u != nullptr;
  const R ra = move ? R(A.st.alpha[l]) : R(0);
  if (PCG && !A.st.active_next[l]) {
    // a load stopped by this iteration's test still takes its last displacement update
    if (move && A.st.stopped[l]) {
      const X* __restrict__ pp = reinterpret_cast<const X*>(A.p + off);
      X* __restrict__ up = reinterpret_cast<X*>(A.u + off);
      for (int h = threadIdx.x; h < C::PLANE / 2; h += T) {
        const X po = pp[h], uo = up[h];
        up[h] = c2(fma(ra, po.x, uo.x), fma(ra, po.y, uo.y));
      }
    }
    return;
  }
  // the half spectrum of the plane stays in flight through the mean and beta reductions
  StageIn<N * C::M, T, X> in;
  StageIn<N, T, X> nyq, twl;
  const X* __restrict__ spec = A.spec + int64_t(l) * 3 * C::NF;
  in.load(spec + (int64_t(c) * N + z) * (N * C::M), [](int e) { return e; });
  nyq.load(spec + Spec<N>::MAIN + (int64_t(c) * N + z) * N, [](int e) { return e; });
  twl.load(A.twy, [](int e) { return e; });
  const int NSLOT = PCG ? A.st.zrows[l] : A.zslots;
  // per-load partials are laid out with the geometry's chunk count (slices of a set are offset by it)
  const double* pgl = A.pg + int64_t(l) * A.f.nkb * N * 4;
  // the output is the next direction p = z + beta p (z alone right after init or without a direction input)
  // (dir: the preconditioner apply that writes the direction in the drop-in layout)
  constexpr bool dir = MODE == kFxyiDir;
  const bool update = dir || (PCG && A.p != nullptr && !A.st.first[l]);
  double mean = 0.0, beta = 0.0;
  if (A.shat || update) {
    // one pass: r.z (offset 0) and this component's s.w (offset 1 + c) partials
    const int off[2] = {0, 1 + c};
    double sums[2] = {0.0, 0.0};
    // (FP64 holds too many of its loads in registers here to share the sums: 128^3 three loads 249 against 208 us)
    if (C::SHARED_SUMS && sizeof(R) == 4) {
      for (int k = threadIdx.x; k < NSLOT; k += T) {
        sums[0] += pgl[4 * k];
        sums[1] += pgl[4 * k + 1 + c];
      }
      block_sums<2>(sums, reinterpret_cast<double*>(tw + N));
    } else {
      wave_reduce_partials_n<2>(pgl, off, NSLOT, 4, sums);
    }
    if (A.shat) mean = sums[1] / double(NN);
    if (dir) {
      beta = sums[0] / fmax(*A.rz_old, 1e-30);
      if (threadIdx.x == 0 && z == 0 && c == 0) *A.rz_out = sums[0];
    } else if (update) {
      const double rz = A.st.rz[l];
      beta = sums[0] / (rz != 0.0 ? rz : 1.0);
    }
  }
  in.store(plane, [](int e) { return e / C::M * C::RS + e % C::M; });
  nyq.store(plane, [](int y) { return y * C::RS + C::M; });
  twl.store(tw);
  // output streams: every load of a chunk is issued before the first use; in
  // FP32 the first chunk is issued before the inverse transforms and stays in
  // flight while they run (FP64, and planes of more than one chunk, lack the
  // registers for that)
  constexpr bool EARLY = sizeof(R) == 4 && C::ITER == C::CH;
  const int64_t soff = (int64_t(design_of(l, A.group)) * 3 + c) * NN + int64_t(z) * C::PLANE;
  const X* __restrict__ sp = reinterpret_cast<const X*>(A.s + soff);
  const X* __restrict__ pp = PCG && A.p != nullptr ? reinterpret_cast<const X*>(A.p + off) : nullptr;
  X* __restrict__ up = move ? reinterpret_cast<X*>(A.u + off) : nullptr;
  X* __restrict__ zp = reinterpret_cast<X*>(A.zout + off);
  const bool scaled = A.s != nullptr;
  // the preconditioner pass also reads s and writes z in the drop-in layout (A.soa == 0): xyz triples per node
  const bool aos = !PCG && !A.soa;
  const int64_t aoff = int64_t(z) * C::PLANE * 3 + c;
  const R* __restrict__ s_aos = aos && scaled ? A.s + int64_t(design_of(l, A.group)) * 3 * NN + aoff : nullptr;
  R* __restrict__ out_aos = dir ? reinterpret_cast<R*>(A.pdir) : A.zout;
  R* __restrict__ z_aos = aos && out_aos ? out_aos + int64_t(l) * 3 * NN + aoff : nullptr;
  // FP32 apply of FP64 vectors: z is written in FP64
  double* __restrict__ z64 = sizeof(R) == 4 && aos && A.zout64 ? A.zout64 + int64_t(l) * 3 * NN + aoff : nullptr;
  const R m = R(mean), tb = R(beta);
  X vs[C::CH], vp[C::CH], vu[C::CH];
  auto load_chunk = [&](int i0) {
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      vs[i] = c2(R(1), R(1));
      vp[i] = c2(R(0), R(0));
      vu[i] = c2(R(0), R(0));
    }
    if (scaled) {
#pragma unroll
      for (int i = 0; i < C::CH; ++i) {
        const int h = pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1);
        if (aos) {
          const R* q = s_aos + 6 * int64_t(h);
          vs[i] = c2(q[0], q[3]);
        } else {
          vs[i] = sp[h];
        }
      }
    }
    if (dir) {
#pragma unroll
      for (int i = 0; i < C::CH; ++i) {
        const R* q = z_aos + 6 * int64_t(pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1));
        vp[i] = c2(q[0], q[3]);
      }
    } else if (update || move) {
#pragma unroll
      for (int i = 0; i < C::CH; ++i) vp[i] = pp[pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1)];
    }
    if (move) {
#pragma unroll
      for (int i = 0; i < C::CH; ++i) vu[i] = up[pair_of<N>(i0 + i < C::ITER ? i0 + i : C::ITER - 1)];
    }
  };
  if (EARLY) load_chunk(0);
  __syncthreads();
  sfft<true, N, typename C::Cols, T, PLAN>(plane, tw, 1);
  constexpr int HALF = C::M / 2, PAIRS = N * (HALF + 1);
  for (int b = threadIdx.x; b < PAIRS; b += T) {
    const int row = b / (HALF + 1), k = b % (HALF + 1);
    X* L = plane + row * C::RS;
    X xk = L[k], xm = L[C::M - k];
    if (k == 0) {
      xk.y = R(0);
      xm.y = R(0);
    }
    const X wk = conjd(tw[k]);
    const X e1 = c2(xk.x + xm.x, xk.y - xm.y);
    const X o1 = cmul(c2(xk.x - xm.x, xk.y + xm.y), wk);
    const X zk = c2(e1.x - o1.y, e1.y + o1.x);
    if (k != 0 && C::M - k != k) {
      const X wm = conjd(tw[C::M - k]);
      const X e2 = c2(xm.x + xk.x, xm.y - xk.y);
      const X o2 = cmul(c2(xm.x - xk.x, xm.y + xk.y), wm);
      L[C::M - k] = c2(e2.x - o2.y, e2.y + o2.x);
    }
    L[k] = zk;
  }
  __syncthreads();
  sfft<true, C::M, typename C::Rows, T, PLAN>(plane, tw, 2);
#pragma unroll
  for (int i0 = 0; i0 < C::ITER; i0 += C::CH) {
    if (!(EARLY && i0 == 0)) load_chunk(i0);
#pragma unroll
    for (int i = 0; i < C::CH; ++i) {
      const int h = int(threadIdx.x) + (i0 + i) * T;
      if (i0 + i >= C::ITER || (!C::EXACT && h >= C::HALF)) continue;
      const int e = 2 * h;
      const int x = e % N, y = e / N;
      const X w = plane[y * C::RS + x / 2];
      X v = scaled ? c2(vs[i].x * w.x - m, vs[i].y * w.y - m) : w;
      if (update) v = c2(fma(tb, vp[i].x, v.x), fma(tb, vp[i].y, v.y));
      if (z64) {
        double* q = z64 + 6 * int64_t(h);
        q[0] = double(v.x);
        q[3] = double(v.y);
      } else if (aos) {
        R* q = z_aos + 6 * int64_t(h);
        q[0] = v.x;
        q[3] = v.y;
      } else {
        zp[h] = v;
      }
      if (move) up[h] = c2(fma(ra, vp[i].x, vu[i].x), fma(ra, vp[i].y, vu[i].y));
    }
  }
}

// ------------------------------------------------------------------ dispatch
template <typename K>
int allow_lds_static(K kernel, size_t bytes) {
  if (bytes <= 65536) return PGJ_OK;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(bytes));
  if (e != hipSuccess) {
    set_error("cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
    return PGJ_ERR_HIP;
  }
  return PGJ_OK;
}

template <int N, typename R>
int fxy_static_n(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
  using C = Cube<N>;
  const size_t lds = C::lds_xy(sizeof(cplx<R>));
  dim3 grid(N, 3, L), block(C::TXY);
  switch (mode) {
    case kFxyScale:
      if (int e = allow_lds_static((fxy_static<N, kFxyScale, R, default_plan<N>()>), lds)) return e;
      hipLaunchKernelGGL((fxy_static<N, kFxyScale, R, default_plan<N>()>), grid, block, lds, s, A);
      break;
    case kFxyPre:
      if (int e = allow_lds_static((fxy_static<N, kFxyPre, R, default_plan<N>()>), lds)) return e;
      hipLaunchKernelGGL((fxy_static<N, kFxyPre, R, default_plan<N>()>), grid, block, lds, s, A);
      break;
    default:
      if (plan_of<N, R>(0) == 1) {
        if (int e = allow_lds_static(fxy_static<N, kFxyPCG, R, 1>, lds)) return e;
        hipLaunchKernelGGL((fxy_static<N, kFxyPCG, R, 1>), grid, block, lds, s, A);
      } else {
        if (int e = allow_lds_static(fxy_static<N, kFxyPCG, R>, lds)) return e;
        hipLaunchKernelGGL((fxy_static<N, kFxyPCG, R>), grid, block, lds, s, A);
      }
  }
  PGJ_LAUNCHED("fxy_static");
  return PGJ_OK;
}

template <int N, typename R, int KC>
int fz_static_kc(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
  using Z = ZPass<N, R, KC>;
  const size_t lds = Z::lds;
  // the per-block partials are laid out for the geometry's chunk count
  PGJ_REQUIRE(Z::BLOCKS <= A.f.nkb * N, "z pass blocks (%d) exceed the partial layout (%d)", Z::BLOCKS, A.f.nkb * N);
  dim3 grid(Z::BLOCKS, 1, L), block(Z::TZ);
  switch (mode) {
    case kFzScale:
      if (int e = allow_lds_static(fz_static<N, kFzScale, R, KC, default_plan<N>()>, lds)) return e;
      hipLaunchKernelGGL((fz_static<N, kFzScale, R, KC, default_plan<N>()>), grid, block, lds, s, A);
      break;
    case kFzPre:
      if (int e = allow_lds_static(fz_static<N, kFzPre, R, KC, default_plan<N>()>, lds)) return e;
      hipLaunchKernelGGL((fz_static<N, kFzPre, R, KC, default_plan<N>()>), grid, block, lds, s, A);
      break;
    case kFzInit:
      if (int e = allow_lds_static(fz_static<N, kFzInit, R, KC, default_plan<N>()>, lds)) return e;
      hipLaunchKernelGGL((fz_static<N, kFzInit, R, KC, default_plan<N>()>), grid, block, lds, s, A);
      break;
    default:
      if (plan_of<N, R>(1) == 1) {
        if (int e = allow_lds_static(fz_static<N, kFzPCG, R, KC, 1>, lds)) return e;
        hipLaunchKernelGGL((fz_static<N, kFzPCG, R, KC, 1>), grid, block, lds, s, A);
      } else {
        if (int e = allow_lds_static(fz_static<N, kFzPCG, R, KC>, lds)) return e;
        hipLaunchKernelGGL((fz_static<N, kFzPCG, R, KC>), grid, block, lds, s, A);
      }
  }
  PGJ_LAUNCHED("fz_static");
  return PGJ_OK;
}

template <int N, typename R, int EU, bool SCALED>
int fz_reg_launch(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
  constexpr size_t lds = ZReg<N>::template lds<R>();
  PGJ_REQUIRE(ZReg<N>::BLOCKS <= A.f.nkb * N, "z pass blocks (%d) exceed the partial layout (%d)", ZReg<N>::BLOCKS,
              A.f.nkb * N);
  const dim3 grid(ZReg<N>::BLOCKS, 1, L), block(64);
  switch (mode) {
    case kFzScale: hipLaunchKernelGGL((fz_reg<N, kFzScale, R, EU, false>), grid, block, lds, s, A); break;
    case kFzPre: hipLaunchKernelGGL((fz_reg<N, kFzPre, R, EU, SCALED>), grid, block, lds, s, A); break;
    case kFzInit: hipLaunchKernelGGL((fz_reg<N, kFzInit, R, EU, SCALED>), grid, block, lds, s, A); break;
    default: hipLaunchKernelGGL((fz_reg<N, kFzPCG, R, EU, SCALED>), grid, block, lds, s, A);
  }
  PGJ_LAUNCHED("fz_reg");
  return PGJ_OK;
}

template <int N, typename R>
int fz_static_n(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
  using W = ZWidths<N, R>;
  if constexpr (zreg<N>()) {
    constexpr int waves = sizeof(R) == 8 ? (N > 64 ? 1 : 2) : N > 64 ? 2 : 3;
    if (A.zkc == 0)
      return A.shat ? fz_reg_launch<N, R, waves, true>(A, L, mode, s) : fz_reg_launch<N, R, waves, false>(A, L, mode, s);
  }
  if constexpr (W::wide != W::def) {
    if (A.zkc == W::wide) return fz_static_kc<N, R, W::wide>(A, L, mode, s);
  }
  return fz_static_kc<N, R, W::def>(A, L, mode, s);
}

// CUs of the current device, cached per device; 0 if the query fails.
static int device_cus() {
  static int cache[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cache[dev] == 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    cache[dev] = cus;
  }
  return cache[dev];
}

bool zpass_wide(const pgj_grid& g, int L, int es) {
  if (es != 8 || !static_cube(g) || g.nx != 64 || L < 1) return false;
  const int64_t cus = device_cus();
  using Zn = ZPass<64, double, ZWidths<64, double>::wide>;
  return cus > 0 && int64_t(Zn::BLOCKS) * L > cus * Zn::per_cu;
}

// The z pass of a workspace: 0 = in registers (fz_reg), else the chunk width of the LDS pass. In registers by default
// wherever the columns divide into its waves; the LDS pass by an explicit radix plan (1 or 3), for the ragged cube, and for
// one FP64 load at 64^3, whose 264 waves leave most SIMDs idle on a long chain of their own. That exception is a table of
// one entry, not a criterion: the other lone loads are faster in registers but for 32^3 FP64, where the two differ by 3 %.
// Graph-replayed launches of one, three and six loads, LDS -> registers (us): 32^3 FP64 6.2 / 7.2 / 9.2 -> 6.4 / 6.5 / 7.0,
// 48^3 FP64 8.4 / 12.9 / 18.8 -> 7.4 / 11.7 / 16.1, 64^3 FP64 11.9 / 20.5 / 30.6 -> 13.3 / 18.7 / 26.1, 64^3 FP32
// 9.5 / 15.4 / 23.8 -> 8.8 / 12.8 / 18.4, 96^3 FP64 31.7 / 68.6 / 127 -> 28.2 / 60.9 / 114, 96^3 FP32 23.7 / 43 / 73 ->
// 23.3 / 34.4 / 63.8, 128^3 FP64 61 / 151 / 295 -> 58 / 140 / 275, 128^3 FP32 49 / 99 / 175 -> 38 / 79 / 163.
template <int N, typename R>
static int zkc_of(const pgj_grid& g, int L) {
  using W = ZWidths<N, R>;
  const int plan = fft_plan(N, int(sizeof(R)), 1);
  if (zreg<N>() && (plan == 2 || (plan == 0 && !(N == 64 && sizeof(R) == 8 && L == 1)))) return 0;
  return W::wide != W::def && zpass_wide(g, L, int(sizeof(R))) ? W::wide : W::def;
}

template <typename R>
void zpass_choose(FFTArgsT<R>& A, const pgj_grid& g, int L) {
  if (!static_cube(g)) {
    A.zkc = runtime_chunk(A.f, L);
    A.zslots = (g.ny * A.f.nkx + A.zkc - 1) / A.zkc;
    return;
  }
  switch (g.nx) {
    case 16: A.zkc = zkc_of<16, R>(g, L); break;
    case 24: A.zkc = zkc_of<24, R>(g, L); break;
    case 32: A.zkc = zkc_of<32, R>(g, L); break;
    case 48: A.zkc = zkc_of<48, R>(g, L); break;
    case 64: A.zkc = zkc_of<64, R>(g, L); break;
    case 96: A.zkc = zkc_of<96, R>(g, L); break;
    default: A.zkc = zkc_of<128, R>(g, L); break;
  }
  A.zslots = A.zkc == 0 ? g.nx / 16 * g.nx + g.nx / 8 : g.nx / 2 / A.zkc * g.nx + g.nx / A.zkc;
}
template void zpass_choose<double>(FFTArgsT<double>&, const pgj_grid&, int);
template void zpass_choose<float>(FFTArgsT<float>&, const pgj_grid&, int);

}  // namespace pgj

extern "C" int pgj_zpass_wide(const pgj_grid* g, int L, int es) {
  return g && L >= 1 && pgj::zpass_wide(*g, L, es) ? 1 : 0;
}

namespace pgj {

template <int N, typename R>
int fxyi_static_n(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
  using C = Cube<N>;
  const size_t lds = C::lds_xy(sizeof(cplx<R>));
  if constexpr (sizeof(R) == 8) {
    if (mode == kFxyiDir) {
      if (int e = allow_lds_static(fxyi_static<N, kFxyiDir, R, default_plan<N>()>, lds)) return e;
      hipLaunchKernelGGL((fxyi_static<N, kFxyiDir, R, default_plan<N>()>), dim3(N, 3, L), dim3(C::TXY), lds, s, A);
      PGJ_LAUNCHED("fxyi_static");
      return PGJ_OK;
    }
  }
  if (mode == kFxyiPre) {
    if (int e = allow_lds_static(fxyi_static<N, kFxyiPre, R, default_plan<N>()>, lds)) return e;
    hipLaunchKernelGGL((fxyi_static<N, kFxyiPre, R, default_plan<N>()>), dim3(N, 3, L), dim3(C::TXY), lds, s, A);
  } else if (plan_of<N, R>(2) == 1) {
    if (int e = allow_lds_static(fxyi_static<N, kFxyiPCG, R, 1>, lds)) return e;
    hipLaunchKernelGGL((fxyi_static<N, kFxyiPCG, R, 1>), dim3(N, 3, L), dim3(C::TXY), lds, s, A);
  } else {
    if (int e = allow_lds_static(fxyi_static<N, kFxyiPCG, R>, lds)) return e;
    hipLaunchKernelGGL((fxyi_static<N, kFxyiPCG, R>), dim3(N, 3, L), dim3(C::TXY), lds, s, A);
  }
  PGJ_LAUNCHED("fxyi_static");
  return PGJ_OK;
}

bool static_fft(const pgj_grid& g) { return static_cube(g); }

#define PGJ_STATIC_SWITCH(CALL)                                       \
  switch (A.nx) {                                                     \
    case 16: return CALL(16);                                         \
    case 24: return CALL(24);                                         \
    case 32: return CALL(32);                                         \
    case 48: return CALL(48);                                         \
    case 64: return CALL(64);                                         \
    case 96: return CALL(96);                                         \
    case 128: return CALL(128);                                       \
    default: set_error("no static FFT for n=%d", A.nx); return PGJ_ERR_UNSUPPORTED; \
  }

template <typename R>
int launch_fxy_static(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
#define CALL(n) fxy_static_n<n, R>(A, L, mode, s)
  PGJ_STATIC_SWITCH(CALL)
#undef CALL
}

template <typename R>
int launch_fz_static(FFTArgsT<R>& A, int L, int mode, hipStream_t s) {
#define CALL(n) fz_static_n<n, R>(A, L, mode, s)
  PGJ_STATIC_SWITCH(CALL)
#undef CALL
}

template <typename R>
int launch_fxyi_static(FFTArgsT<R>& A, int L, hipStream_t s, int mode) {
#define CALL(n) fxyi_static_n<n, R>(A, L, mode, s)
  PGJ_STATIC_SWITCH(CALL)
#undef CALL
}

template int launch_fxy_static<double>(FFTArgsT<double>&, int, int, hipStream_t);
template int launch_fz_static<double>(FFTArgsT<double>&, int, int, hipStream_t);
template int launch_fxyi_static<double>(FFTArgsT<double>&, int, hipStream_t, int);
template int launch_fxy_static<float>(FFTArgsT<float>&, int, int, hipStream_t);
template int launch_fz_static<float>(FFTArgsT<float>&, int, int, hipStream_t);
template int launch_fxyi_static<float>(FFTArgsT<float>&, int, hipStream_t, int);

}  // namespace pgj
