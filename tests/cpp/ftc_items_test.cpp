// Host-side test of the FT convolution's rows per item: the fewest rows whose items all run at once on the device's
// CUs, 16 where no count does, and every row in exactly one item.
#include <cstdio>
#include <vector>

#include "fdas_kernels.h"
#include "fdas_plan.h"

using namespace fdas;

int main() {
  int failures = 0;
  for (uint32_t tile : {1024u, 2048u, 4096u})
    for (uint32_t n_cu : {32u, 64u, 256u})  // a device in parts, and a whole one
      for (uint32_t n_bins : {999u, 4999u, 32768u, 131072u, 700001u})
        for (uint32_t T : {1u, 33u, 85u, 255u}) {
          const uint32_t max_taps = 421, slots = ftconv_slots(tile, n_cu);
          if (slots != n_cu * 4 * 3 * 64 / (tile / 16)) ++failures, std::printf("FAIL slots %u %u\n", tile, n_cu);
          std::vector<uint32_t> taps(T);
          for (uint32_t t = 0; t < T; ++t) taps[t] = 1 + 420 * (t > T / 2 ? t - T / 2 : T / 2 - t) / (T / 2 + 1);
          const std::vector<FtcJob> wide = plan_ftc_rows(tile, n_bins, max_taps, taps, 0, T, 64);
          auto items = [&](uint32_t target) {
            uint64_t n = 0;
            for (const FtcJob& j : wide) {
              const uint32_t rows = ftc_rows_per_item(j.n_rows, target);
              n += uint64_t(j.n_tiles) * ((j.n_rows + rows - 1) / rows);
            }
            return n;
          };
          uint32_t want = 1;
          while (want < kFtcRowsPerItem && items(want) > slots) ++want;
          std::vector<FtcJob> jobs = wide;
          fit_ftc_items(jobs, slots);
          for (const FtcJob& j : jobs)
            if (j.rows_per_item != ftc_rows_per_item(j.n_rows, want) || j.n_chunks * j.rows_per_item < j.n_rows ||
                (j.n_chunks - 1) * j.rows_per_item >= j.n_rows)
              ++failures, std::printf("FAIL tile %u, %u CUs, %u bins, %u rows\n", tile, n_cu, n_bins, T);
        }
  if (failures == 0) std::printf("ftc items test ok\n");
  return failures != 0;
}
