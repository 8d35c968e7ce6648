// Host-side test of the front end's twiddle tables: for every length, the tables its transforms read, and no others.
#include <cmath>
#include <cstdio>

#include "fdas_plan.h"

using namespace fdas;

int main() {
  int failures = 0;
  const double pi = 3.14159265358979323846;
  for (uint32_t log2n = 1; log2n <= 22; ++log2n) {
    const uint32_t n = 1u << log2n, n1 = n <= 4096 ? 1u : 1u << (log2n / 2), n2 = n / n1;
    const LineTables t = line_tables({n1, n2});
    size_t want = 0;
    for (int i = 0; i < 2; ++i) {
      const uint32_t L = i == 0 ? n1 : n2, NT = L / 16, D = NT / 16;
      const bool reads1 = L > 16, reads2 = L > 256;
      if (i == 0 || n1 != n2) want += (reads1 ? L : 0) + (reads2 ? NT : 0);
      double err = 0;
      for (uint32_t k = 0; k < 16 && reads1; ++k)
        for (uint32_t b = 0; b < NT; ++b) {
          if (t.w1[i] + L > t.data.size()) return std::printf("FAIL table 1 of %u outside\n", L), 1;
          const float2 v = t.data[t.w1[i] + k * NT + b];
          err = std::fmax(err, std::hypot(v.x - std::cos(2 * pi * b * k / L), v.y + std::sin(2 * pi * b * k / L)));
        }
      for (uint32_t k = 0; k < 16 && reads2; ++k)
        for (uint32_t d = 0; d < D; ++d) {
          if (t.w2[i] + NT > t.data.size()) return std::printf("FAIL table 2 of %u outside\n", L), 1;
          const float2 v = t.data[t.w2[i] + k * D + d];
          err = std::fmax(err, std::hypot(v.x - std::cos(2 * pi * d * k / NT), v.y + std::sin(2 * pi * d * k / NT)));
        }
      if (err > 1e-7) ++failures, std::printf("FAIL length %u: error %g\n", L, err);
    }
    if (t.data.size() != want) ++failures, std::printf("FAIL N %u: %zu entries, %zu are read\n", n, t.data.size(), want);
  }
  if (failures == 0) std::printf("line tables test ok\n");
  return failures != 0;
}
