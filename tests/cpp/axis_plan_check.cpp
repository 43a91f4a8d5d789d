// Host check of the runtime FFT's axis plans: every supported length factors into its stages, a group of lanes covers
// every stage's butterflies, and the multiply-shift divisions are exact over the ranges the kernels use them on. Also
// the LDS and partial-row bounds of every supported box whose axes come from a list of lengths.
#include <cstdio>

#include "../../partial-green-jacobi_amd/csrc/layout.h"

using namespace pgj;

#define CHECK(c, ...)                     \
  do {                                    \
    if (!(c)) {                           \
      std::printf("failed: %s: ", #c);    \
      std::printf(__VA_ARGS__);           \
      std::printf("\n");                  \
      return 1;                           \
    }                                     \
  } while (0)

static bool smooth(int n) {
  for (int p : {2, 3, 5, 7})
    while (n % p == 0) n /= p;
  return n == 1;
}

int main() {
  for (int n = 1; n <= kMaxAxis; ++n) {
    const AxisPlan& a = axis_plan(n);
    CHECK((a.count >= 0) == smooth(n), "%d", n);
    if (a.count < 0) continue;
    int product = 1;
    CHECK(a.n == n && a.G >= 1 && a.lpw >= 1 && a.G * a.lpw <= 64, "%d", n);
    for (int s = 0; s < a.count; ++s) {
      const AxisPlan::Stage& st = a.st[s];
      CHECK(st.R >= 2 && st.R <= 10 && st.Ns == product && st.nb * st.R == n && st.tws * st.Ns * st.R == n, "%d", n);
      CHECK(st.nb <= a.G * (st.R == 3 ? 2 : 1), "%d stage %d", n, s);
      for (int j = 0; j < st.nb; ++j) CHECK(int((unsigned(j) * st.mNs) >> 16) == j / st.Ns, "%d %d", n, j);
      product *= st.R;
    }
    CHECK(product == n, "%d", n);
    for (int lane = 0; lane < 64; ++lane) {
      CHECK(int((lane * a.mG) >> 16) == lane / a.G, "%d %d", n, lane);
      CHECK(int((lane * a.mL) >> 16) == lane / a.lpw, "%d %d", n, lane);
    }
    if (n > 1)
      for (uint64_t x = 0; x < 65536; ++x) CHECK(int((x * magic32(n)) >> 32) == int(x) / n, "%d", n);
  }
  int boxes = 0;
  for (int nz : {2, 45, 100, 243, 256})
    for (int ny = 2; ny <= kMaxAxis; ++ny)
      for (int nx = 2; nx <= kMaxAxis; ++nx) {
        pgj_grid g{};
        g.nz = nz; g.ny = ny; g.nx = nx;
        const FFTGeom f = fft_geom(g);
        if (!f.runtime_ok || static_cube(g)) continue;
        ++boxes;
        CHECK(32 * 8 + (size_t(ny) * f.rs + nx + ny) * 16 <= 148 * 1024, "%d %d", ny, nx);
        CHECK((ny * f.nkx + kMinChunk - 1) / kMinChunk <= f.nkb * ny, "%d %d", ny, nx);
        CHECK(ny * nx < 65536 && ny * f.rs < 65536, "%d %d", ny, nx);
      }
  std::printf("%d boxes\nOK\n", boxes);
  return 0;
}
