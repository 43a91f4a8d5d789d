// HEX8 operator kernels: the row-march apply (drop-in and fused PCG form),
// the independent thread-per-node reference apply, rhs, energies, C^H,
// mean stress, nodal diagonal / partial Green-Jacobi scale and projection.
#include <cmath>
#include <mutex>
#include <type_traits>

#include "hex8_kernels.h"

namespace pgj {

// Raw inputs of one node row segment (the input vector: u, or the PCG direction p).
template <int MODE, int R, int XPL, typename T>
struct Rows {
  T v[R + 1][XPL][3];
};

// Row-march HEX8 apply. Lanes map to x (XPL consecutive x per lane), each of
// the W row-waves marches R element rows over the z-layers of the block, a
// halo wave computes the element row below the block, and contributions to a
// neighbour wave's first node row go through a double-buffered LDS slot. The
// next plane's inputs are fetched before the current layer is computed.
// PLANE selects the plane-carry march: the in-plane butterflies of each node
// plane are computed once and shared by the two element layers that touch it
// (forward: the top plane of layer z is the bottom plane of layer z+1;
// transposed: the modal forces of both layers on a plane are summed before
// one in-plane transform), which halves the in-plane butterflies, the x
// neighbour exchanges and the LDS traffic per element.
template <int MODE, int XPL, int R, bool CUBIC, int MAXT, typename T, bool PLANE>
__global__ __launch_bounds__(MAXT) void hex8_rowmarch(RowArgsT<T> A) {
  // the drop-in apply works on AoS vectors, the resident iteration on SoA
  constexpr bool SOA = MODE == kModePCG;
  constexpr unsigned ES = sizeof(T);
  extern __shared__ __align__(16) unsigned char smem[];
  T* lds = reinterpret_cast<T*>(smem);
  const int lane = threadIdx.x & 63;
  // wave index and everything derived from it are wave-uniform: keep them in SGPRs
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int l = blockIdx.z;
  const T* __restrict__ mat = A.a + size_t(design_of(l, A.group)) * A.N;
  const RowMarch& c = A.cfg;
  const int W = c.W;
  const int nx = A.nx, ny = A.ny, nz = A.nz;
  const unsigned N = unsigned(A.N);
  // XCD-aware row groups: workgroups are dealt to the 8 XCDs round robin by
  // linear id, so when the row-group count is a multiple of 8 each XCD gets a
  // contiguous range of row groups, and the halo row a block reads has just
  // been fetched into the same L2 by its neighbour.
  const int nrg = int(gridDim.x);
  const int rg = nrg % 8 == 0 ? int(blockIdx.x % 8) * (nrg / 8) + int(blockIdx.x / 8) : int(blockIdx.x);
  const int y0 = rg * W * R, z0 = blockIdx.y * c.ZC;
  const int xl = lane % c.nl;
  const bool lane_on = lane < c.nl;
  const unsigned xo = unsigned(xl * XPL);

  if (MODE == kModePCG) {
    if (!A.st.active[l]) return;
  } else if (A.mask && !A.mask[l]) {
    // Inactive load: zeros, as the reference's pre-zeroed output.
    T* o = A.out + size_t(l) * 3 * N;
    if (wave < W && lane_on) {
      for (int j = 0; j < R; ++j)
        for (int zi = 0; zi < c.ZC; ++zi)
          for (int xi = 0; xi < XPL; ++xi) {
            const unsigned node = unsigned((z0 + zi) * ny + (y0 + wave * R + j)) * unsigned(nx) + xo + xi;
            for (int d = 0; d < 3; ++d) o[3 * node + d] = T(0);
          }
    }
    return;
  }

  const bool halo = wave == W;
  const int ybase = halo ? y0 - 1 : y0 + wave * R;
  const int rows = halo ? 1 : R;  // element rows computed by this wave
  // uniform base pointers per component (SoA) or per load (AoS)
  const T* __restrict__ in = A.u + size_t(l) * 3 * N;
  T* __restrict__ out = A.out + size_t(l) * 3 * N;
  // element offsets in bytes (32-bit): uniform base + 32-bit offset selects the SGPR-base addressing form
  auto at = [&](unsigned node, int d) -> unsigned { return ES * (SOA ? unsigned(d) * N + node : 3u * node + unsigned(d)); };
  auto ld = [](const T* base, unsigned off) -> T {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
  };
  auto st = [](T* base, unsigned off, T v) { *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off) = v; };
  auto row_of = [&](int plane, int j) -> unsigned {
    return unsigned(plane * ny + wrapi(ybase + j, ny)) * unsigned(nx);
  };

  auto fetch = [&](int plane, Rows<MODE, R, XPL, T>& dst, T (&arow)[R][XPL]) {
#pragma unroll
    for (int j = 0; j <= R; ++j) {
      if (j > rows) break;
      const unsigned rb = row_of(plane, j);
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi) {
        const unsigned node = rb + xo + xi;
#pragma unroll
        for (int d = 0; d < 3; ++d) dst.v[j][xi][d] = ld(in, at(node, d));
        if (j < R) arow[j][xi] = ld(mat, ES * node);
      }
    }
  };
  // Node values of a fetched plane.
  auto settle = [&](const Rows<MODE, R, XPL, T>& src, T (&dst)[R + 1][XPL][3]) {
#pragma unroll
    for (int j = 0; j <= R; ++j) {
      if (j > rows) break;
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
        for (int d = 0; d < 3; ++d) dst[j][xi][d] = src.v[j][xi][d];
    }
  };

  double pq = 0.0;
  const int src_right = (xl + 1) % c.nl;       // lane holding x + XPL
  const int src_left = (xl + c.nl - 1) % c.nl;  // lane holding x - 1
  if constexpr (PLANE) {
    T nodeU[R + 1][XPL][3];
    // bottom-plane nodes of the owned rows for p.q: held, or (two FP64 x per lane) read again from the cache, because
    // the registers they take would spill
    constexpr bool RELOAD = XPL == 2 && sizeof(T) == 8;
    T nodeLo[R][XPL][3];
    T PL[R][XPL][3][4];              // in-plane modes of the bottom plane, per element column
    T CM[R][XPL][3][4];              // modal forces on the bottom plane from the layer below
    T accL[R + 1][XPL][3];
    T aL[R][XPL], aU[R][XPL], aN[R][XPL];
    const int slot_size = (c.W + 1) * 64 * 3 * XPL;
    // in-plane modes of every element column of the rows this wave computes
    auto plane_modes = [&](const T (&nd)[R + 1][XPL][3], T (&P)[R][XPL][3][4]) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (j >= rows) break;
        T nb[2][3];
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
#pragma unroll
          for (int d = 0; d < 3; ++d) nb[oy][d] = __shfl(nd[j + oy][0][d], src_right, 64);
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
          for (int d = 0; d < 3; ++d)
            plane_forward(nd[j][xi][d], xi + 1 < XPL ? nd[j][xi + 1][d] : nb[0][d], nd[j + 1][xi][d],
                          xi + 1 < XPL ? nd[j + 1][xi + 1][d] : nb[1][d], P[j][xi][d]);
      }
    };
    Rows<MODE, R, XPL, T> raw;
    fetch(wrapi(z0 - 1, nz), raw, aL);
    settle(raw, nodeU);
    plane_modes(nodeU, PL);
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          nodeLo[j][xi][d] = nodeU[j][xi][d];
#pragma unroll
          for (int m = 0; m < 4; ++m) CM[j][xi][d][m] = T(0);
        }
    fetch(z0, raw, aU);
    for (int li = 0; li <= c.ZC; ++li) {
      const int zl = wrapi(z0 - 1 + li, nz), zu = wrapi(z0 + li, nz);
      settle(raw, nodeU);
      if (li < c.ZC) fetch(wrapi(z0 + li + 1, nz), raw, aN);  // prefetch the next plane
#pragma unroll
      for (int j = 0; j <= R; ++j)
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
          for (int d = 0; d < 3; ++d) accL[j][xi][d] = T(0);
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (j >= rows) break;
        T nb[2][3];
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
#pragma unroll
          for (int d = 0; d < 3; ++d) nb[oy][d] = __shfl(nodeU[j + oy][0][d], src_right, 64);
        T spill[2][3];  // contributions of this lane's last element column to x + 1 (next lane)
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi) {
          T PU[3][4], Um[3][8], F[3][8];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            plane_forward(nodeU[j][xi][d], xi + 1 < XPL ? nodeU[j][xi + 1][d] : nb[0][d], nodeU[j + 1][xi][d],
                          xi + 1 < XPL ? nodeU[j + 1][xi + 1][d] : nb[1][d], PU[d]);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              Um[d][m] = PL[j][xi][d][m] + PU[d][m];
              Um[d][m | 4] = PU[d][m] - PL[j][xi][d][m];
            }
          }
          hex8_modal_core<CUBIC, T>(Um, aL[j][xi], A.coef, F);
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            T M[4], f[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              M[m] = CM[j][xi][d][m] + (F[d][m] - F[d][m | 4]);
              CM[j][xi][d][m] = F[d][m] + F[d][m | 4];
              PL[j][xi][d][m] = PU[d][m];
            }
            plane_transposed(M, f);
            accL[j][xi][d] += f[0];
            accL[j + 1][xi][d] += f[2];
            if (xi + 1 < XPL) {
              accL[j][xi + 1][d] += f[1];
              accL[j + 1][xi + 1][d] += f[3];
            } else {
              spill[0][d] = f[1];
              spill[1][d] = f[3];
            }
          }
        }
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
#pragma unroll
          for (int d = 0; d < 3; ++d) accL[j + oy][0][d] += __shfl(spill[oy][d], src_left, 64);
      }
      // Export the contributions to the first node row of the next wave.
      T* slots = lds + (li & 1) * slot_size;
      T* slot = slots + wave * 64 * 3 * XPL;
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
        for (int d = 0; d < 3; ++d) slot[(xi * 3 + d) * 64 + lane] = halo ? accL[1][xi][d] : accL[R][xi][d];
      __syncthreads();
      if (!halo) {
        const T* from = slots + (wave == 0 ? W : wave - 1) * 64 * 3 * XPL;
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
          for (int d = 0; d < 3; ++d) accL[0][xi][d] += from[(xi * 3 + d) * 64 + lane];
        if (li >= 1 && lane_on) {
#pragma unroll
          for (int j = 0; j < R; ++j) {
            const unsigned rb = unsigned(zl * ny + ybase + j) * unsigned(nx);
#pragma unroll
            for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
              for (int d = 0; d < 3; ++d) {
                st(out, at(rb + xo + xi, d), accL[j][xi][d]);
                if (MODE != kModeApply) {
                  const T own = RELOAD ? ld(in, at(rb + xo + xi, d)) : nodeLo[j][xi][d];
                  pq = fma(double(own), double(accL[j][xi][d]), pq);
                }
              }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi) {
#pragma unroll
          for (int d = 0; d < 3; ++d) nodeLo[j][xi][d] = nodeU[j][xi][d];
          aL[j][xi] = aU[j][xi];
          aU[j][xi] = aN[j][xi];
        }
    }
    if (MODE != kModeApply) {
      const double total = block_sum(pq, reinterpret_cast<double*>(lds + 2 * slot_size));
      if (threadIdx.x == 0) A.ppq[int64_t(l) * A.ppq_stride + blockIdx.y * gridDim.x + rg] = total;
    }
    return;
  } else {
  T nodeL[R + 1][XPL][3], nodeU[R + 1][XPL][3];
  T carry[R][XPL][3];
  T accL[R + 1][XPL][3], accU[R + 1][XPL][3];
  T aL[R][XPL], aU[R][XPL], aN[R][XPL];
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
      for (int d = 0; d < 3; ++d) carry[j][xi][d] = T(0);

  const int slot_size = (c.W + 1) * 64 * 6 * XPL;

  Rows<MODE, R, XPL, T> raw;
  fetch(wrapi(z0 - 1, nz), raw, aL);
  settle(raw, nodeL);
  fetch(z0, raw, aU);
  for (int li = 0; li <= c.ZC; ++li) {
    const int zl = wrapi(z0 - 1 + li, nz), zu = wrapi(z0 + li, nz);
    settle(raw, nodeU);
    if (li < c.ZC) fetch(wrapi(z0 + li + 1, nz), raw, aN);  // prefetch the next plane
#pragma unroll
    for (int j = 0; j <= R; ++j)
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          accL[j][xi][d] = (j < R) ? carry[j][xi][d] : T(0);
          accU[j][xi][d] = T(0);
        }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (j >= rows) break;
      // Right neighbours (x + XPL) of the four node rows this element row touches.
      T nb[2][2][3];
#pragma unroll
      for (int oy = 0; oy < 2; ++oy)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          nb[oy][0][d] = __shfl(nodeL[j + oy][0][d], src_right, 64);
          nb[oy][1][d] = __shfl(nodeU[j + oy][0][d], src_right, 64);
        }
      T spill[2][2][3];  // contributions of this lane's last element to x + 1 (next lane)
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi) {
        T ue[24], fe[24];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int ox = n & 1, oy = (n >> 1) & 1, oz = (n >> 2) & 1;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            T v;
            if (ox == 0 || xi + 1 < XPL) {
              const int xs = xi + ox;
              v = oz ? nodeU[j + oy][xs][d] : nodeL[j + oy][xs][d];
            } else {
              v = nb[oy][oz][d];
            }
            ue[3 * n + d] = v;
          }
        }
        hex8_element<CUBIC, T>(ue, aL[j][xi], A.coef, fe);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int ox = n & 1, oy = (n >> 1) & 1, oz = (n >> 2) & 1;
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const T v = fe[3 * n + d];
            if (ox == 0) {
              if (oz) accU[j + oy][xi][d] += v; else accL[j + oy][xi][d] += v;
            } else if (xi + 1 < XPL) {
              if (oz) accU[j + oy][xi + 1][d] += v; else accL[j + oy][xi + 1][d] += v;
            } else {
              spill[oy][oz][d] = v;
            }
          }
        }
      }
#pragma unroll
      for (int oy = 0; oy < 2; ++oy)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          accL[j + oy][0][d] += __shfl(spill[oy][0][d], src_left, 64);
          accU[j + oy][0][d] += __shfl(spill[oy][1][d], src_left, 64);
        }
    }
    // Export the contributions to the first node row of the next wave.
    T* slots = lds + (li & 1) * slot_size;
    T* slot = slots + wave * 64 * 6 * XPL;
#pragma unroll
    for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        slot[(xi * 6 + d) * 64 + lane] = halo ? accL[1][xi][d] : accL[R][xi][d];
        slot[(xi * 6 + 3 + d) * 64 + lane] = halo ? accU[1][xi][d] : accU[R][xi][d];
      }
    __syncthreads();
    if (!halo) {
      const T* from = slots + (wave == 0 ? W : wave - 1) * 64 * 6 * XPL;
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          accL[0][xi][d] += from[(xi * 6 + d) * 64 + lane];
          accU[0][xi][d] += from[(xi * 6 + 3 + d) * 64 + lane];
        }
      if (li >= 1 && lane_on) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const unsigned rb = unsigned(zl * ny + ybase + j) * unsigned(nx);
#pragma unroll
          for (int xi = 0; xi < XPL; ++xi) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
              st(out, at(rb + xo + xi, d), accL[j][xi][d]);
              if (MODE != kModeApply) pq = fma(double(nodeL[j][xi][d]), double(accL[j][xi][d]), pq);
            }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < R; ++j)
#pragma unroll
        for (int xi = 0; xi < XPL; ++xi)
#pragma unroll
          for (int d = 0; d < 3; ++d) carry[j][xi][d] = accU[j][xi][d];
    }
#pragma unroll
    for (int j = 0; j <= R; ++j)
#pragma unroll
      for (int xi = 0; xi < XPL; ++xi) {
#pragma unroll
        for (int d = 0; d < 3; ++d) nodeL[j][xi][d] = nodeU[j][xi][d];
        if (j < R) {
          aL[j][xi] = aU[j][xi];
          aU[j][xi] = aN[j][xi];
        }
      }
  }
  if (MODE != kModeApply) {
    const double total = block_sum(pq, reinterpret_cast<double*>(lds + 2 * slot_size));
    if (threadIdx.x == 0) A.ppq[int64_t(l) * A.ppq_stride + blockIdx.y * gridDim.x + rg] = total;
  }
  }
}

// The 24x24 element stiffness of C0 by its tensor-product form, independent of the modal form of the other kernels.
// The integrals over the element factor into per-axis ones over two ends. With the displacements written as the node's
// own value and differences along the axes to the other ends, each factor is one over both ends (`sum`) or one of the
// other end alone: mass h / 2 and h / 6, stiffness 0 and -1 / h, derivative of the node's function s and s / 2, of the
// other's 0 and -s / 2, with s = -1 or +1 the node's end. So K_ii and K_ij take, for the set of axes `o` along which a
// quantity is a difference,
//   diag[i][o],  -s_i s_j (lam [j in o] + mu [i in o]) / (2 or, with both, 4) mass_k   (i != j, k the third axis):
// 39 numbers, all held in scalar registers. The node's own value (o empty) drops out exactly.
struct RefStiffness {
  double diag[3][8];
  double lam[3][2], mu[3][2], both[3][2];   // lam / 2, mu / 2 and (lam + mu) / 4 times the mass along k
};

// Certification apply. A thread owns the column of nodes (x, y) over ZC planes and marches them: it loads each plane's
// 3 x 3 neighbours once, turns them into differences from the column's node, and adds their terms to the forces of the
// four elements of the layer below and of the layer above on the layer's two nodes of the column: 456 FMAs and 31 loads
// per node, with nine fixed offsets per thread. Bound by FP64 issue at two waves per SIMD. One load at 64^3 15 us, six 57,
// 128^3 six 383; eight whole elements evaluated per node for 3 of their 24 forces each took 39, 195 and 1562.
// The differences also keep the digits: products with whole displacements (17, 62 and 388 us) cancel the rigid part only
// in the rounded sum. Relative error on a smooth field plus an offset of 0 and 3, at 32^3: 9.8e-16 and 9.7e-14, of the
// modal row march 6.6e-16 and 5.2e-14, here 2.6e-16 and 2.5e-16; at 9 x 5 x 64 1.2e-15 and 9.4e-14, 2.8e-16 and 8.0e-15,
// 2.7e-16 and 2.7e-16.
// I: unsigned where the byte offsets of a vector fit 32 bits (uniform base + 32-bit offset), else int64_t.
template <bool CERT, typename I>
__global__ __launch_bounds__(256) void hex8_reference(RefArgs A, RefStiffness K, int ZC) {
  __shared__ double red[8];
  const int l = blockIdx.y;
  const int64_t P = int64_t(A.nx) * A.ny;
  const int64_t id = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int z0 = int(id / P) * ZC, z1 = min(z0 + ZC, A.nz);
  double res2 = 0.0;
  if (z0 < A.nz) {
    const int col = int(id % P), x = col % A.nx, y = col / A.nx;
    const int xs[3] = {wrapi(x - 1, A.nx), x, wrapi(x + 1, A.nx)};
    const int ys[3] = {wrapi(y - 1, A.ny), y, wrapi(y + 1, A.ny)};
    const double* __restrict__ mat = A.a + int64_t(design_of(l, A.group)) * A.N;
    const double* __restrict__ u = A.u + int64_t(l) * 3 * A.N;
    const double* __restrict__ rhs = CERT ? A.rhs + int64_t(l) * 3 * A.N : nullptr;
    double* __restrict__ out = A.out + int64_t(l) * 3 * A.N;
    const I cs = A.soa ? I(A.N) : I(1), ns = A.soa ? I(1) : I(3);   // strides of components and nodes
    // a plane's values: the column's node, its differences to x - 1, x + 1, y - 1, y + 1, and the mixed differences of
    // the four quadrants e (bit set: the minus side of the axis)
    double q[9][3], zq[9][3];     // of this plane; of the plane below, then differences of the two
    // forces, for a = 1, of the layer's elements on its bottom and top node of the column: the terms of single differences
    // ([0], the largest) and of mixed ones ([1]) are summed apart, so that fewer sums round at the size of the force
    double bot[2][4][3], top[2][4][3];
    double carry[3] = {0.0, 0.0, 0.0};
    // terms of the plane's values (SZ = 0) or of the differences along z (SZ = 1) on the layer's node at z corner ZN
    auto add = [&](auto sz, auto zn, const double (&w)[9][3], double (&force)[2][4][3]) {
      constexpr int SZ = decltype(sz)::value, ZN = decltype(zn)::value;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int sxy = 0; sxy < 4; ++sxy) {
          if (SZ == 0 && sxy == 0) continue;
          const int at = sxy == 0 ? 0 : sxy == 1 ? 2 - (e & 1) : sxy == 2 ? 4 - (e >> 1) : 5 + e;
          const int o = sxy | SZ << 2, n = e | ZN << 2;   // n: the node is the corner of the element's bits
          const bool flip = SZ == 1 && ZN == 1;           // the other end of the top node lies below
          double (&f)[4][3] = force[(o & (o - 1)) != 0];
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            f[e][a] = fma(flip ? -K.diag[a][o] : K.diag[a][o], w[at][a], f[e][a]);
#pragma unroll
            for (int b = 0; b < 3; ++b) {
              const int k = 3 - a - b;
              if (b == a || !((o >> a | o >> b) & 1)) continue;
              const int m = (o >> k) & 1;
              const double c = !((o >> a) & 1) ? K.lam[k][m] : !((o >> b) & 1) ? K.mu[k][m] : K.both[k][m];
              f[e][a] = fma((((n >> a ^ n >> b) & 1) != 0) != flip ? c : -c, w[at][b], f[e][a]);
            }
          }
        }
    };
    using Z0 = std::integral_constant<int, 0>;
    using Z1 = std::integral_constant<int, 1>;
    I at[3][3];
#pragma unroll
    for (int py = 0; py < 3; ++py)
#pragma unroll
      for (int px = 0; px < 3; ++px) at[py][px] = I(ys[py]) * I(A.nx) + I(xs[px]);
#pragma unroll 1
    for (int z = z0 - 1; z <= z1; ++z) {
      const I plane = I(wrapi(z, A.nz)) * I(P), below = I(wrapi(z - 1, A.nz)) * I(P);
#pragma unroll
      for (int py = 0; py < 3; ++py)
#pragma unroll
        for (int px = 0; px < 3; ++px)
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            const int to = px == 1 && py == 1 ? 0 : py == 1 ? (px == 0 ? 1 : 2) : px == 1 ? (py == 0 ? 3 : 4)
                                                 : 5 + (px == 0 ? 1 : 0) + (py == 0 ? 2 : 0);
            q[to][d] = u[ns * (plane + at[py][px]) + cs * I(d)];
          }
#pragma unroll
      for (int d = 0; d < 3; ++d) {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[5 + e][d] -= q[4 - (e >> 1)][d];   // along x, in the rows y - 1 and y + 1
#pragma unroll
        for (int i = 1; i < 5; ++i) q[i][d] -= q[0][d];
#pragma unroll
        for (int e = 0; e < 4; ++e) q[5 + e][d] -= q[2 - (e & 1)][d];
      }
      if (z >= z0) {
        double ae[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) ae[e] = mat[below + at[1 - (e >> 1)][1 - (e & 1)]];
#pragma unroll
        for (int i = 0; i < 9; ++i)
#pragma unroll
          for (int d = 0; d < 3; ++d) zq[i][d] = q[i][d] - zq[i][d];
        add(Z1{}, Z0{}, zq, bot);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int d = 0; d < 3; ++d) top[0][e][d] = top[1][e][d] = 0.0;
        add(Z0{}, Z1{}, q, top);
        add(Z1{}, Z1{}, zq, top);
        if (z > z0) {
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            double acc = carry[d];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = fma(ae[e], bot[0][e][d] + bot[1][e][d], acc);
            const I idx = ns * (below + at[1][1]) + cs * I(d);
            if (CERT) {
              const double r = rhs[idx] - acc;
              out[idx] = r;
              res2 = fma(r, r, res2);
            } else {
              out[idx] = acc;
            }
          }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          carry[d] = 0.0;
#pragma unroll
          for (int e = 0; e < 4; ++e) carry[d] = fma(ae[e], top[0][e][d] + top[1][e][d], carry[d]);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int d = 0; d < 3; ++d) bot[0][e][d] = bot[1][e][d] = 0.0;
      add(Z0{}, Z0{}, q, bot);
#pragma unroll
      for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int d = 0; d < 3; ++d) zq[i][d] = q[i][d];
    }
  }
  if (CERT) {
    const double t = block_sum(res2, red);
    if (threadIdx.x == 0) A.pres[(int64_t(l) * A.pres_rows + blockIdx.x) * 4 + 3] = t;
  }
}

// Per-block component sums of a (L, 3N) vector into partial rows of 4 doubles.
__device__ __forceinline__ int64_t lidx(int soa, int l, int d, int64_t i, int64_t N) {
  return soa ? (int64_t(l) * 3 + d) * N + i : (int64_t(l) * N + i) * 3 + d;
}

__global__ __launch_bounds__(256) void component_sums(const double* v, int64_t N, double* part, int soa) {
  __shared__ double red[8];
  const int l = blockIdx.y;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double s[3] = {0.0, 0.0, 0.0};
  if (i < N)
    for (int d = 0; d < 3; ++d) s[d] = v[lidx(soa, l, d, i, N)];
  for (int d = 0; d < 3; ++d) {
    const double t = block_sum(s[d], red);
    if (threadIdx.x == 0) part[(int64_t(l) * gridDim.x + blockIdx.x) * 4 + d] = t;
  }
}

// v -= mean per load/component (mean from component_sums partials; the first
// wave reduces them in a fixed order and shares the result through LDS).
// FINISHED: component_means has left the means in the load's first partial row.
template <bool FINISHED>
__global__ __launch_bounds__(256) void subtract_mean(double* v, int64_t N, const double* part, int nblk, int soa) {
  __shared__ double mean[3];
  const int l = blockIdx.y;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (FINISHED) {
    if (threadIdx.x < 3) mean[threadIdx.x] = part[int64_t(l) * nblk * 4 + threadIdx.x];
  } else if (threadIdx.x < 64) {
    const double* p = part + int64_t(l) * nblk * 4;
    for (int d = 0; d < 3; ++d) {
      const double s = wave_reduce_partials(p + d, nblk, 4);
      if (threadIdx.x == 0) mean[d] = s / double(N);
    }
  }
  __syncthreads();
  if (i < N)
    for (int d = 0; d < 3; ++d) v[lidx(soa, l, d, i, N)] -= mean[d];
}

// The three means of load blockIdx.x into slots 0..2 of its first partial row, which only this block reads.
__global__ __launch_bounds__(256) void component_means(int64_t N, double* part, int nblk) {
  __shared__ double red[12];
  double* p = part + int64_t(blockIdx.x) * nblk * 4;
  double s[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
  for (int b = threadIdx.x; b < nblk; b += 256)
    for (int d = 0; d < 3; ++d) s[d] += p[int64_t(b) * 4 + d];
  block_sums<3>(s, red);
  if (threadIdx.x == 0)
    for (int d = 0; d < 3; ++d) p[d] = s[d] / double(N);
}

// AoS (L, N, 3) <-> SoA (L, 3, N)
__global__ __launch_bounds__(256) void transpose_kernel(const double* in, double* out, int64_t N, int to_soa) {
  const int l = blockIdx.y;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  for (int d = 0; d < 3; ++d) {
    if (to_soa) out[lidx(1, l, d, i, N)] = in[lidx(0, l, d, i, N)];
    else out[lidx(0, l, d, i, N)] = in[lidx(1, l, d, i, N)];
  }
}

// ------------------------------------------------------------------------ rhs
// f_node = -sum_{8 elements} a_e V Bbar_a^T C0 eps with centroid gradients +-1/(4h).
__global__ __launch_bounds__(256) void hex8_rhs_kernel(int nz, int ny, int nx, ElementCoef c, const double* a,
                                                       double m0, double m1, double m2, double m3, double m4,
                                                       double m5, double* out, int soa) {
  const int64_t N = int64_t(nx) * ny * nz;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const int x = int(i % nx), y = int((i / nx) % ny), z = int(i / (int64_t(nx) * ny));
  // C0 eps (Voigt, engineering shear)
  const double tr = m0 + m1 + m2;
  const double s0 = c.lam * tr + 2 * c.mu * m0, s1 = c.lam * tr + 2 * c.mu * m1, s2 = c.lam * tr + 2 * c.mu * m2;
  const double s3 = c.mu * m3, s4 = c.mu * m4, s5 = c.mu * m5;
  double f[3] = {0.0, 0.0, 0.0};
  for (int o = 0; o < 8; ++o) {
    const int ex = wrapi(x - (o & 1), nx), ey = wrapi(y - ((o >> 1) & 1), ny), ez = wrapi(z - ((o >> 2) & 1), nz);
    const double ae = a[(int64_t(ez) * ny + ey) * nx + ex] * c.vol;
    const double dx = (o & 1) ? c.g[0] : -c.g[0];
    const double dy = (o & 2) ? c.g[1] : -c.g[1];
    const double dz = (o & 4) ? c.g[2] : -c.g[2];
    f[0] -= ae * (dx * s0 + dy * s5 + dz * s4);
    f[1] -= ae * (dx * s5 + dy * s1 + dz * s3);
    f[2] -= ae * (dx * s4 + dy * s3 + dz * s2);
  }
  for (int d = 0; d < 3; ++d) out[lidx(soa, 0, d, i, N)] = f[d];
}

// Affine element displacement chi_n,d = (E * (offset_n * h))_d for a macro strain.
__device__ __forceinline__ void affine_local(const double* m, const ElementCoef& c, double (&chi)[24]) {
  const double h[3] = {1.0 / (4.0 * c.g[0]), 1.0 / (4.0 * c.g[1]), 1.0 / (4.0 * c.g[2])};
  const double E[3][3] = {{m[0], 0.5 * m[5], 0.5 * m[4]}, {0.5 * m[5], m[1], 0.5 * m[3]}, {0.5 * m[4], 0.5 * m[3], m[2]}};
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const double p[3] = {(n & 1) * h[0], ((n >> 1) & 1) * h[1], ((n >> 2) & 1) * h[2]};
#pragma unroll
    for (int d = 0; d < 3; ++d) chi[3 * n + d] = E[d][0] * p[0] + E[d][1] * p[1] + E[d][2] * p[2];
  }
}

struct MacroSet {
  double m[6][6];
};

struct DiagTable {
  double v[8][3];
};

__device__ __forceinline__ void gather_element(const double* u, int nz, int ny, int nx, int x, int y, int z,
                                               double (&ue)[24]) {
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    const int xx = wrapi(x + (n & 1), nx), yy = wrapi(y + ((n >> 1) & 1), ny), zz = wrapi(z + ((n >> 2) & 1), nz);
    const int64_t node = (int64_t(zz) * ny + yy) * nx + xx;
#pragma unroll
    for (int d = 0; d < 3; ++d) ue[3 * n + d] = u[3 * node + d];
  }
}

template <bool CUBIC>
__global__ __launch_bounds__(256) void hex8_energy_kernel(int nz, int ny, int nx, ElementCoef c, const double* u,
                                                          MacroSet ms, double* out) {
  const int64_t N = int64_t(nx) * ny * nz;
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int l = blockIdx.y;
  if (e >= N) return;
  const int x = int(e % nx), y = int((e / nx) % ny), z = int(e / (int64_t(nx) * ny));
  double ue[24], fe[24], chi[24];
  gather_element(u + int64_t(l) * 3 * N, nz, ny, nx, x, y, z, ue);
  affine_local(ms.m[l], c, chi);
#pragma unroll
  for (int k = 0; k < 24; ++k) ue[k] += chi[k];
  hex8_element<CUBIC>(ue, 1.0, c, fe);
  double en = 0.0;
#pragma unroll
  for (int k = 0; k < 24; ++k) en = fma(ue[k], fe[k], en);
  out[int64_t(l) * N + e] = en / c.vol;
}

// C^H partials: per block the 21 upper-triangle sums of a_e (Ke v_i) . v_j / V over 256 elements, 32 at a time. Thread
// (load i, element) gathers v_i, evaluates Ke v_i once and shares v_i through LDS; the pairs (i, i + 0..3 mod 6) are
// its dot products (i + 3 for i < 3), which covers every pair once. One thread per element with all pairs gathered the
// element's displacements 27 times (64^3: 88 us, 128^3 670 us).
constexpr int kEffElements = 32, kEffThreads = 6 * kEffElements;

template <bool CUBIC>
__global__ __launch_bounds__(kEffThreads) void effective_partials(int nz, int ny, int nx, ElementCoef c, const double* a,
                                                                  const double* u6, double* part) {
  __shared__ double v[6][24][kEffElements];
  const int64_t N = int64_t(nx) * ny * nz;
  const int i = threadIdx.x / kEffElements, k = threadIdx.x % kEffElements;
  double m[6], s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int q = 0; q < 6; ++q) m[q] = q == i ? 1.0 : 0.0;
  double chi[24];
  affine_local(m, c, chi);
  for (int g = 0; g < 256; g += kEffElements) {
    const int64_t e = int64_t(blockIdx.x) * 256 + g + k;
    const int64_t ec = e < N ? e : N - 1;
    const int x = int(ec % nx), y = int((ec / nx) % ny), z = int(ec / (int64_t(nx) * ny));
    const double ae = e < N ? a[ec] : 0.0;
    double vi[24], fi[24];
    gather_element(u6 + int64_t(i) * 3 * N, nz, ny, nx, x, y, z, vi);
#pragma unroll
    for (int q = 0; q < 24; ++q) vi[q] += chi[q];
    hex8_element<CUBIC>(vi, 1.0, c, fi);
    __syncthreads();   // the previous group's values have been read
#pragma unroll
    for (int q = 0; q < 24; ++q) v[i][q][k] = vi[q];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int j = i + p < 6 ? i + p : i + p - 6;
      double t = 0.0;
#pragma unroll
      for (int q = 0; q < 24; ++q) t = fma(fi[q], v[j][q][k], t);
      s[p] = e < N ? s[p] + ae * t / c.vol : s[p];
    }
  }
  // sums over the 32 lanes of a load
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int off = kEffElements / 2; off >= 1; off >>= 1) s[p] += __shfl_xor(s[p], off, 64);
  if (k == 0)
    for (int p = 0; p < (i < 3 ? 4 : 3); ++p) {
      const int j = i + p < 6 ? i + p : i + p - 6, lo = min(i, j), hi = max(i, j);
      part[int64_t(blockIdx.x) * 21 + lo * 6 - lo * (lo - 1) / 2 + (hi - lo)] = s[p];
    }
}

__global__ void effective_finish(const double* part, int nblk, int64_t N, double* out) {
  const int idx = blockIdx.x;  // one wavefront per upper-triangle entry
  const double s = wave_reduce_partials(part + idx, nblk, 21);
  if (threadIdx.x != 0) return;
  int k = 0;
  for (int i = 0; i < 6; ++i)
    for (int j = i; j < 6; ++j, ++k)
      if (k == idx) {
        out[i * 6 + j] = s / double(N);
        out[j * 6 + i] = s / double(N);
      }
}

__global__ __launch_bounds__(256) void avg_stress_partials(int nz, int ny, int nx, ElementCoef c, const double* a,
                                                           const double* u, MacroSet ms, double* part) {
  __shared__ double red[8];
  const int64_t N = int64_t(nx) * ny * nz;
  const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double sig[6] = {0, 0, 0, 0, 0, 0};
  if (e < N) {
    const int x = int(e % nx), y = int((e / nx) % ny), z = int(e / (int64_t(nx) * ny));
    double eps[6];
    for (int k = 0; k < 6; ++k) eps[k] = ms.m[0][k];
    for (int n = 0; n < 8; ++n) {
      const int xx = wrapi(x + (n & 1), nx), yy = wrapi(y + ((n >> 1) & 1), ny), zz = wrapi(z + ((n >> 2) & 1), nz);
      const int64_t node = (int64_t(zz) * ny + yy) * nx + xx;
      const double ux = u[3 * node], uy = u[3 * node + 1], uz = u[3 * node + 2];
      const double dx = (n & 1) ? c.g[0] : -c.g[0], dy = (n & 2) ? c.g[1] : -c.g[1], dz = (n & 4) ? c.g[2] : -c.g[2];
      eps[0] += dx * ux;
      eps[1] += dy * uy;
      eps[2] += dz * uz;
      eps[3] += dz * uy + dy * uz;
      eps[4] += dz * ux + dx * uz;
      eps[5] += dy * ux + dx * uy;
    }
    const double ae = a[e];
    const double tr = eps[0] + eps[1] + eps[2];
    for (int k = 0; k < 3; ++k) sig[k] = ae * (c.lam * tr + 2 * c.mu * eps[k]);
    for (int k = 3; k < 6; ++k) sig[k] = ae * c.mu * eps[k];
  }
  for (int k = 0; k < 6; ++k) {
    const double t = block_sum(sig[k], red);
    if (threadIdx.x == 0) part[int64_t(blockIdx.x) * 6 + k] = t;
  }
}

__global__ void avg_stress_finish(const double* part, int nblk, int64_t N, double* out) {
  const int k = blockIdx.x;
  const double s = wave_reduce_partials(part + k, nblk, 6);
  if (threadIdx.x == 0) out[k] = s / double(N);
}

// Nodal diagonal: d_i = sum_o a_{i-o} diag(Ke)[o]; log partials for the scale.
__global__ __launch_bounds__(256) void diagonal_kernel(int nz, int ny, int nx, const double* a, DiagTable ed,
                                                       double* d, double* logpart) {
  __shared__ double red[8];
  const int64_t N = int64_t(nx) * ny * nz;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  double lsum = 0.0;
  if (i < N) {
    const int x = int(i % nx), y = int((i / nx) % ny), z = int(i / (int64_t(nx) * ny));
    double acc[3] = {0.0, 0.0, 0.0};
    for (int o = 0; o < 8; ++o) {
      const int ex = wrapi(x - (o & 1), nx), ey = wrapi(y - ((o >> 1) & 1), ny), ez = wrapi(z - ((o >> 2) & 1), nz);
      const double ae = a[(int64_t(ez) * ny + ey) * nx + ex];
      for (int k = 0; k < 3; ++k) acc[k] += ae * ed.v[o][k];
    }
    for (int k = 0; k < 3; ++k) {
      if (d) d[3 * i + k] = acc[k];
      lsum += log(acc[k]);
    }
  }
  const double t = block_sum(lsum, red);
  if (threadIdx.x == 0) logpart[blockIdx.x] = t;
}

__global__ __launch_bounds__(256) void scale_kernel(int nz, int ny, int nx, const double* a, DiagTable ed,
                                                    double alpha_value, const double* alpha_dev, const double* logpart,
                                                    int nblk, double* s, int soa) {
  // alpha from device memory (an on-device selection) when given
  const double alpha = alpha_dev ? *alpha_dev : alpha_value;
  __shared__ double smean;
  const int64_t N = int64_t(nx) * ny * nz;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (threadIdx.x < 64) {
    const double tot = wave_reduce_partials(logpart, nblk, 1);
    if (threadIdx.x == 0) smean = tot / double(3 * N);
  }
  __syncthreads();
  const double mean = smean;
  if (i >= N) return;
  const int x = int(i % nx), y = int((i / nx) % ny), z = int(i / (int64_t(nx) * ny));
  double acc[3] = {0.0, 0.0, 0.0};
  for (int o = 0; o < 8; ++o) {
    const int ex = wrapi(x - (o & 1), nx), ey = wrapi(y - ((o >> 1) & 1), ny), ez = wrapi(z - ((o >> 2) & 1), nz);
    const double ae = a[(int64_t(ez) * ny + ey) * nx + ex];
    for (int k = 0; k < 3; ++k) acc[k] += ae * ed.v[o][k];
  }
  for (int k = 0; k < 3; ++k) s[lidx(soa, 0, k, i, N)] = exp(-0.5 * alpha * (log(acc[k]) - mean));
}


// ------------------------------------------------------------------ launchers

bool cubic(const pgj_grid& g) { return g.hx == g.hy && g.hy == g.hz; }

ElementCoef coef_of(const pgj_grid& g) { return make_coef(g.hx, g.hy, g.hz, g.lam, g.mu); }

DiagTable diag_table(const pgj_grid& g) {
  DiagTable t{};
  ElementCoef c = coef_of(g);
  for (int k = 0; k < 24; ++k) {
    double u[24] = {0}, f[24];
    u[k] = 1.0;
    hex8_element<false>(u, 1.0, c, f);
    t.v[k / 3][k % 3] = f[k];
  }
  return t;
}

int check_grid(const pgj_grid* g) {
  PGJ_REQUIRE(g != nullptr, "null grid");
  PGJ_REQUIRE(g->nx >= 2 && g->ny >= 2 && g->nz >= 2, "grid dimensions must be >= 2, got (%d,%d,%d)", g->nz, g->ny,
              g->nx);
  PGJ_REQUIRE(g->hx > 0 && g->hy > 0 && g->hz > 0, "positive voxel sizes required");
  PGJ_REQUIRE(int64_t(g->nx) * g->ny * g->nz < (int64_t(1) << 31) / 3, "grid too large");
  return PGJ_OK;
}

template <int MODE, int XPL, int R, int MAXT, bool PLANE, typename T>
int launch_rowmarch_t(const pgj_grid& g, int L, RowArgsT<T>& A, hipStream_t s) {
  const RowMarch& c = A.cfg;
  dim3 grid(c.by, c.bz, L), block(64 * (c.W + 1));
  const size_t lds = 2 * size_t(c.W + 1) * 64 * (PLANE ? 3 : 6) * XPL * sizeof(T) + 64 * 8;
  if (cubic(g))
    hipLaunchKernelGGL((hex8_rowmarch<MODE, XPL, R, true, MAXT, T, PLANE>), grid, block, lds, s, A);
  else
    hipLaunchKernelGGL((hex8_rowmarch<MODE, XPL, R, false, MAXT, T, PLANE>), grid, block, lds, s, A);
  PGJ_LAUNCHED("hex8_rowmarch");
  return PGJ_OK;
}

template <int MODE, typename T>
int launch_rowmarch_m(const pgj_grid& g, int L, RowArgsT<T>& A, hipStream_t s) {
  const RowMarch& c = A.cfg;
  constexpr int kPlaneThreads = sizeof(T) == 8 ? 320 : 576;
  if (c.plane) {
    if (c.xpl == 1) return launch_rowmarch_t<MODE, 1, 1, kPlaneThreads, true>(g, L, A, s);
    return launch_rowmarch_t<MODE, 2, 1, 320, true>(g, L, A, s);
  }
  if (c.R == 2) return launch_rowmarch_t<MODE, 1, 2, 320, false>(g, L, A, s);
  if (c.xpl == 1) return launch_rowmarch_t<MODE, 1, 1, 576, false>(g, L, A, s);
  return launch_rowmarch_t<MODE, 2, 1, 320, false>(g, L, A, s);
}

template <typename T>
int launch_rowmarch(const pgj_grid& g, int L, int mode, RowArgsT<T>& A, hipStream_t s) {
  A.nz = g.nz; A.ny = g.ny; A.nx = g.nx;
  A.N = int64_t(g.nx) * g.ny * g.nz;
  A.cfg = rowmarch_config(g, L, int(sizeof(T)));
  A.coef = coef_of(g);
  if constexpr (sizeof(T) == 8)
    if (mode == kModeApplyDot) return launch_rowmarch_m<kModeApplyDot>(g, L, A, s);
  return mode == kModeApply ? launch_rowmarch_m<kModeApply>(g, L, A, s) : launch_rowmarch_m<kModePCG>(g, L, A, s);
}
template int launch_rowmarch<double>(const pgj_grid&, int, int, RowArgsT<double>&, hipStream_t);
template int launch_rowmarch<float>(const pgj_grid&, int, int, RowArgsT<float>&, hipStream_t);

// The numbers of the element stiffness (RefStiffness).
static RefStiffness ref_stiffness(const pgj_grid& g) {
  RefStiffness K{};
  const double h[3] = {g.hx, g.hy, g.hz};
  auto mass = [&](int axis, int other) { return other ? h[axis] / 6 : h[axis] / 2; };
  for (int o = 0; o < 8; ++o) {
    double grad[3];   // of the two nodes' derivatives along one axis
    for (int j = 0; j < 3; ++j) {
      grad[j] = (o >> j) & 1 ? -1.0 / h[j] : 0.0;
      for (int k = 0; k < 3; ++k)
        if (k != j) grad[j] *= mass(k, (o >> k) & 1);
    }
    for (int i = 0; i < 3; ++i) {
      K.diag[i][o] = g.lam * grad[i];
      for (int j = 0; j < 3; ++j) K.diag[i][o] += g.mu * (i == j ? 2.0 : 1.0) * grad[j];
    }
  }
  for (int k = 0; k < 3; ++k)
    for (int other = 0; other < 2; ++other) {
      K.lam[k][other] = 0.5 * g.lam * mass(k, other);
      K.mu[k][other] = 0.5 * g.mu * mass(k, other);
      K.both[k][other] = 0.25 * (g.lam + g.mu) * mass(k, other);
    }
  return K;
}

// Planes per thread: the longest march that leaves 96k threads (six waves per CU), so that one layer in ZC + 1 is
// redundant; at least 2.
static int reference_zc(const pgj_grid& g, int L) {
  const int64_t N = int64_t(g.nx) * g.ny * g.nz;
  int zc = 16;
  while (zc > 2 && N * L / zc < 98304) zc /= 2;
  return zc;
}

int reference_blocks(const pgj_grid& g, int L) {
  const int zc = reference_zc(g, L);
  return int((int64_t(g.nx) * g.ny * ((g.nz + zc - 1) / zc) + 255) / 256);
}

template <bool CERT>
static int launch_reference_t(const pgj_grid& g, int L, RefArgs& A, hipStream_t s) {
  const dim3 grid(unsigned(reference_blocks(g, L)), L), block(256);
  const RefStiffness K = ref_stiffness(g);
  const int zc = reference_zc(g, L);
  if (A.N < (int64_t(1) << 32) / 24)
    hipLaunchKernelGGL((hex8_reference<CERT, unsigned>), grid, block, 0, s, A, K, zc);
  else
    hipLaunchKernelGGL((hex8_reference<CERT, int64_t>), grid, block, 0, s, A, K, zc);
  PGJ_LAUNCHED("hex8_reference");
  return PGJ_OK;
}

int launch_reference(const pgj_grid& g, int L, RefArgs& A, bool cert, hipStream_t s) {
  A.nz = g.nz; A.ny = g.ny; A.nx = g.nx;
  A.N = int64_t(g.nx) * g.ny * g.nz;
  return cert ? launch_reference_t<true>(g, L, A, s) : launch_reference_t<false>(g, L, A, s);
}

// Where a launch has more than 1400 blocks of loads with more than 256 partial rows each (more than 40^3 nodes), the means
// are reduced once per load instead of once per block, whose reductions grow with the square of the rows. Projection of
// one load, three, six, by the blocks / in a launch before them (us): 64^3 18.2 / 21.0, 29.9 / 25.0, 51.1 / 39.3, 45^3
// 18.2 / 20.6, 18.3 / 20.8, 26.9 / 22.2, 80^3 28.7 / 21.4, 64.8 / 40.2, 121 / 68, 128^3 207 / 52, 621 / 135, 1270 / 319.
int launch_subtract_mean(const pgj_grid& g, int L, double* v, double* part, int soa, hipStream_t s) {
  const int64_t N = int64_t(g.nx) * g.ny * g.nz;
  const int nblk = int((N + 255) / 256);
  if (nblk > 256 && int64_t(nblk) * L > 1400) {
    hipLaunchKernelGGL(component_means, dim3(L), dim3(256), 0, s, N, part, nblk);
    PGJ_LAUNCHED("component_means");
    hipLaunchKernelGGL(subtract_mean<true>, dim3(nblk, L), dim3(256), 0, s, v, N, part, nblk, soa);
  } else {
    hipLaunchKernelGGL(subtract_mean<false>, dim3(nblk, L), dim3(256), 0, s, v, N, part, nblk, soa);
  }
  PGJ_LAUNCHED("subtract_mean");
  return PGJ_OK;
}

int launch_component_sums(const pgj_grid& g, int L, const double* v, double* part, int soa, hipStream_t s) {
  const int64_t N = int64_t(g.nx) * g.ny * g.nz;
  dim3 grid(unsigned((N + 255) / 256), L);
  hipLaunchKernelGGL(component_sums, grid, dim3(256), 0, s, v, N, part, soa);
  PGJ_LAUNCHED("component_sums");
  return PGJ_OK;
}

}  // namespace pgj

using namespace pgj;

extern "C" int pgj_hex8_apply(const pgj_grid* g, int L, const double* a, const double* u, const uint8_t* active,
                              double* out, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && a && u && out, "invalid apply arguments");
  if (!rowmarch_config(*g, L).valid) {
    PGJ_REQUIRE(active == nullptr, "active mask needs the row-march kernel (nx <= 128 and nx %% ceil(nx/64) == 0)");
    return pgj_hex8_apply_reference(g, L, a, u, out, stream);
  }
  RowArgs A{};
  A.a = a; A.u = u; A.out = out; A.mask = active;
  return launch_rowmarch(*g, L, kModeApply, A, as_stream(stream));
}

extern "C" int pgj_hex8_apply32(const pgj_grid* g, int L, const float* a, const float* u, const uint8_t* active,
                                float* out, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && a && u && out, "invalid apply arguments");
  PGJ_REQUIRE(rowmarch_config(*g, L, 4).valid, "the FP32 apply needs the row-march kernel (nx <= 128 and nx %% ceil(nx/64) == 0)");
  RowArgsT<float> A{};
  A.a = a; A.u = u; A.out = out; A.mask = active;
  return launch_rowmarch(*g, L, kModeApply, A, as_stream(stream));
}

extern "C" int pgj_hex8_apply_reference(const pgj_grid* g, int L, const double* a, const double* u, double* out,
                                        void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && a && u && out, "invalid apply arguments");
  RefArgs A{};
  A.a = a; A.u = u; A.out = out;
  return launch_reference(*g, L, A, false, as_stream(stream));
}

extern "C" int pgj_hex8_rhs(const pgj_grid* g, const double* a, const double macro[6], double* out, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(a && macro && out, "invalid rhs arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  hipLaunchKernelGGL(hex8_rhs_kernel, dim3(unsigned((N + 255) / 256)), dim3(256), 0, as_stream(stream), g->nz, g->ny,
                     g->nx, coef_of(*g), a, macro[0], macro[1], macro[2], macro[3], macro[4], macro[5], out, 0);
  PGJ_LAUNCHED("hex8_rhs");
  return PGJ_OK;
}

namespace pgj {

int launch_rhs(const pgj_grid& g, const double* a, const double* macro, double* out, int soa, hipStream_t s) {
  const int64_t N = int64_t(g.nx) * g.ny * g.nz;
  hipLaunchKernelGGL(hex8_rhs_kernel, dim3(unsigned((N + 255) / 256)), dim3(256), 0, s, g.nz, g.ny, g.nx, coef_of(g),
                     a, macro[0], macro[1], macro[2], macro[3], macro[4], macro[5], out, soa);
  PGJ_LAUNCHED("hex8_rhs");
  return PGJ_OK;
}

int launch_scale(const pgj_grid& g, const double* a, double alpha, double* d, double* s_out, double* ws, int soa,
                 hipStream_t s, const double* alpha_dev) {
  const int64_t N = int64_t(g.nx) * g.ny * g.nz;
  const int nblk = int((N + 255) / 256);
  DiagTable t = diag_table(g);
  hipLaunchKernelGGL(diagonal_kernel, dim3(nblk), dim3(256), 0, s, g.nz, g.ny, g.nx, a, t, d, ws);
  PGJ_LAUNCHED("diagonal_kernel");
  hipLaunchKernelGGL(scale_kernel, dim3(nblk), dim3(256), 0, s, g.nz, g.ny, g.nx, a, t, alpha, alpha_dev, ws, nblk,
                     s_out, soa);
  PGJ_LAUNCHED("scale_kernel");
  return PGJ_OK;
}

}  // namespace pgj

extern "C" int pgj_hex8_energy(const pgj_grid* g, int L, const double* u, const double* macros, double* out,
                               void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 6 && u && macros && out, "energy needs 1 <= L <= 6 loads");
  MacroSet ms{};
  for (int l = 0; l < L; ++l)
    for (int k = 0; k < 6; ++k) ms.m[l][k] = macros[6 * l + k];
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  dim3 grid(unsigned((N + 255) / 256), L);
  if (cubic(*g))
    hipLaunchKernelGGL(hex8_energy_kernel<true>, grid, dim3(256), 0, as_stream(stream), g->nz, g->ny, g->nx,
                       coef_of(*g), u, ms, out);
  else
    hipLaunchKernelGGL(hex8_energy_kernel<false>, grid, dim3(256), 0, as_stream(stream), g->nz, g->ny, g->nx,
                       coef_of(*g), u, ms, out);
  PGJ_LAUNCHED("hex8_energy");
  return PGJ_OK;
}

extern "C" size_t pgj_effective_tensor_ws_bytes(const pgj_grid* g) {
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  return align256(size_t((N + 255) / 256) * 21 * 8);
}

extern "C" int pgj_effective_tensor(const pgj_grid* g, const double* a, const double* u6, double* ws, double* out36,
                                    void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(a && u6 && ws && out36, "invalid effective tensor arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  const int nblk = int((N + 255) / 256);
  hipStream_t s = as_stream(stream);
  if (cubic(*g))
    hipLaunchKernelGGL(effective_partials<true>, dim3(nblk), dim3(kEffThreads), 0, s, g->nz, g->ny, g->nx, coef_of(*g), a, u6, ws);
  else
    hipLaunchKernelGGL(effective_partials<false>, dim3(nblk), dim3(kEffThreads), 0, s, g->nz, g->ny, g->nx, coef_of(*g), a, u6,
                       ws);
  PGJ_LAUNCHED("effective_partials");
  hipLaunchKernelGGL(effective_finish, dim3(21), dim3(64), 0, s, ws, nblk, N, out36);
  PGJ_LAUNCHED("effective_finish");
  return PGJ_OK;
}

// ---- C^H without a caller workspace -----------------------------------------------------------------
// The partial sums live in a file-scope device array, one copy per GPU. Host code never passes the array's
// name to a kernel: in host code it is only a stand-in for the symbol. Its device address is looked up once
// per device (hipGetSymbolAddress, with that device current) and kept in `g_scratch_ptr`.
static constexpr int64_t kNoAllocMaxElements = int64_t(1) << 22;                 // 4,194,304 elements
static constexpr size_t kNoAllocScratchDoubles = size_t(kNoAllocMaxElements / 256) * 21;  // 2,752,512 bytes
static __device__ __align__(256) double scratch[kNoAllocScratchDoubles];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

int scratch_for_current_device(double** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("hipGetDevice failed: %s", hipGetErrorString(e));
    return PGJ_ERR_HIP;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("device %d beyond the %d devices the scratch table holds", dev, kMaxDevices);
    return PGJ_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
      return PGJ_ERR_HIP;
    }
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return PGJ_OK;
}
}  // namespace

extern "C" int64_t pgj_effective_tensor_noalloc_max_elements(void) { return kNoAllocMaxElements; }

extern "C" int pgj_effective_tensor_noalloc(const pgj_grid* g, const double* a, const double* u6, double* out36,
                                            void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(a && u6 && out36, "invalid effective tensor arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  PGJ_REQUIRE(N <= kNoAllocMaxElements,
              "pgj_effective_tensor_noalloc: grid of %lld elements exceeds the %lld-element limit of its "
              "built-in scratch; use pgj_effective_tensor with a workspace", (long long)N,
              (long long)kNoAllocMaxElements);
  double* part = nullptr;
  if (int e = scratch_for_current_device(&part)) return e;
  // every block overwrites its own 21 partials before effective_finish reads them: nothing to clear
  const int nblk = int((N + 255) / 256);
  hipStream_t s = as_stream(stream);
  if (cubic(*g))
    hipLaunchKernelGGL(effective_partials<true>, dim3(nblk), dim3(kEffThreads), 0, s, g->nz, g->ny, g->nx, coef_of(*g), a,
                       u6, part);
  else
    hipLaunchKernelGGL(effective_partials<false>, dim3(nblk), dim3(kEffThreads), 0, s, g->nz, g->ny, g->nx, coef_of(*g), a,
                       u6, part);
  PGJ_LAUNCHED("effective_partials");
  hipLaunchKernelGGL(effective_finish, dim3(21), dim3(64), 0, s, part, nblk, N, out36);
  PGJ_LAUNCHED("effective_finish");
  return PGJ_OK;
}

extern "C" size_t pgj_avg_stress_ws_bytes(const pgj_grid* g) {
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  return align256(size_t((N + 255) / 256) * 6 * 8);
}

extern "C" int pgj_hex8_avg_stress(const pgj_grid* g, const double* a, const double* u, const double macro[6],
                                   double* ws, double* out6, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(a && u && macro && ws && out6, "invalid stress arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  const int nblk = int((N + 255) / 256);
  MacroSet ms{};
  for (int k = 0; k < 6; ++k) ms.m[0][k] = macro[k];
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(avg_stress_partials, dim3(nblk), dim3(256), 0, s, g->nz, g->ny, g->nx, coef_of(*g), a, u, ms, ws);
  PGJ_LAUNCHED("avg_stress_partials");
  hipLaunchKernelGGL(avg_stress_finish, dim3(6), dim3(64), 0, s, ws, nblk, N, out6);
  PGJ_LAUNCHED("avg_stress_finish");
  return PGJ_OK;
}

extern "C" size_t pgj_scale_ws_bytes(const pgj_grid* g) {
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  return align256(size_t((N + 255) / 256) * 8);
}

extern "C" int pgj_diagonal_scale(const pgj_grid* g, const double* a, double alpha, double* d, double* s_out,
                                  double* ws, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(a && s_out && ws, "invalid scale arguments");
  return launch_scale(*g, a, alpha, d, s_out, ws, 0, as_stream(stream));
}

extern "C" size_t pgj_project_ws_bytes(const pgj_grid* g, int L) {
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  return align256(size_t(L) * size_t((N + 255) / 256) * 4 * 8);
}

extern "C" int pgj_project(const pgj_grid* g, int L, double* v, double* ws, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && v && ws, "invalid projection arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  const int nblk = int((N + 255) / 256);
  hipStream_t s = as_stream(stream);
  (void)nblk;
  if (int e = launch_component_sums(*g, L, v, ws, 0, s)) return e;
  return launch_subtract_mean(*g, L, v, ws, 0, s);
}

extern "C" int pgj_aos_to_soa(const pgj_grid* g, int L, const double* in, double* out, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && in && out && in != out, "invalid transpose arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  hipLaunchKernelGGL(transpose_kernel, dim3(unsigned((N + 255) / 256), L), dim3(256), 0, as_stream(stream), in, out, N, 1);
  PGJ_LAUNCHED("transpose");
  return PGJ_OK;
}

extern "C" int pgj_soa_to_aos(const pgj_grid* g, int L, const double* in, double* out, void* stream) {
  if (int e = check_grid(g)) return e;
  PGJ_REQUIRE(L >= 1 && L <= 65535 && in && out && in != out, "invalid transpose arguments");
  const int64_t N = int64_t(g->nx) * g->ny * g->nz;
  hipLaunchKernelGGL(transpose_kernel, dim3(unsigned((N + 255) / 256), L), dim3(256), 0, as_stream(stream), in, out, N, 0);
  PGJ_LAUNCHED("transpose");
  return PGJ_OK;
}
