// Host check of the span numbering of the gradient and right-hand-side
// kernels (local-dg_amd/csrc/ldg_kernels.hpp: make_spans, span_elements), built
// with hipcc for the host only by tests/test_spans.py (no GPU needed): over
// meshes of one run and of strips, with ragged last strips and last
// workgroups, every element belongs to exactly one workgroup, at most E per
// workgroup, and the element coordinates and neighbour distances that the
// kernels derive from the element number agree with the periodic mesh.
#include <cstdio>
#include <vector>

#include "ldg_kernels.hpp"

using namespace ldg;

int main() {
  long bad = 0, cases = 0;
  const int sizes[][3] = {{3, 3, 3}, {4, 3, 5}, {8, 8, 8}, {31, 17, 23}, {64, 64, 3}, {64, 63, 4}, {200, 5, 3}, {61, 37, 3}, {40, 70, 4},
                          {3, 200, 3}, {5, 3, 90}, {130, 130, 3}};
  for (int n = 2; n <= 6; ++n)
    for (int E : {1, 2, 3, 4, 5, 7, 8, 14, 16, 32})
      for (const auto &m : sizes) {
        InstDesc d{};
        d.nx = m[0]; d.ny = m[1]; d.nz = m[2];
        d.nelem = (long)m[0] * m[1] * m[2];
        const long nb = make_spans(d, n, E);
        std::vector<int> cnt(d.nelem, 0);
        for (long b = 0; b < nb; ++b) {
          int kl, ne;
          span_elements(d, E, (int)b, kl, ne);
          if (ne < 1 || ne > E) ++bad;
          for (int e = 0; e < ne; ++e) {
            if (kl + e < 0 || kl + e >= d.nelem) { ++bad; continue; }
            cnt[kl + e]++;
          }
        }
        for (long k = 0; k < d.nelem; ++k) {
          if (cnt[k] != 1) ++bad;
          const int x = (int)(k % d.nx), y = (int)(k / d.nx % d.ny), z = (int)(k / d.nx / d.ny);
          int c[3];
          element_coords(d, (int)k, c);
          if (c[0] != x || c[1] != y || c[2] != z) ++bad;
          for (int l = 0; l < 3; ++l) {
            const int p[3] = {l == 0 ? (x + d.nx - 1) % d.nx : x, l == 1 ? (y + d.ny - 1) % d.ny : y,
                              l == 2 ? (z + d.nz - 1) % d.nz : z};
            if (k + neighbor_step(d, c, l, -1) != p[0] + (long)d.nx * (p[1] + (long)d.ny * p[2])) ++bad;
          }
        }
        ++cases;
      }
  std::printf("%ld meshes x workgroup sizes, %ld failures\n%s\n", cases, bad, bad ? "FAILED" : "ok");
  return bad ? 1 : 0;
}
