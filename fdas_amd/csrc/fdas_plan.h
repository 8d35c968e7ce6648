// Host-side planning shared by the single-trial context and the batch/serve engine.
#pragma once

#include <hip/hip_runtime.h>

#include <complex>
#include <cstdint>
#include <vector>

#include "fdas_jobs.h"
#include "fdas_kernels.h"

namespace fdas {

// Rows one FT-convolution work item convolves: enough to amortise the forward
// transform of its tile, small enough for several items per tile.  `target` is
// the preferred count; the rows are split into equal chunks of at most that.
constexpr uint32_t kFtcRowsPerItem = 16;
uint32_t ftc_rows_per_item(uint32_t n_rows, uint32_t target = kFtcRowsPerItem);

// Splits rows [row_begin, row_begin + n_rows) into contiguous groups, each with
// its own overlap (longest non-zero template of the group minus one, rounded up
// to 4).  row_taps may be empty (every row then uses max_taps).  The returned
// jobs have geometry and rows filled; pointers and item_begin are left to the
// caller.  The grouping (and so every FOP value) depends only on the tile, N and
// the tap extents; rows_target only sets how many rows one work item takes.
std::vector<FtcJob> plan_ftc_rows(uint32_t tile, uint32_t n_bins, uint32_t max_taps,
                                  const std::vector<uint32_t>& row_taps, uint32_t row_begin, uint32_t n_rows,
                                  uint32_t max_groups, uint32_t rows_target = kFtcRowsPerItem);

// Fewer rows per item for a launch that would leave CUs idle: the smallest count
// whose items are all resident at once (`slots` workgroups), so that a row's
// latency, not the number of rows in a row, sets the span; launches with more
// items than that at 16 rows keep 16, which spend the fewest forward transforms.
// Measured, us per launch (1 trial), at 16 rows / at the count chosen here:
//   4,999 bins x 33 templates, tile 1024: 26 / 6.6 (1 row)
//   32,768 x 85, tile 1024: 33 / 12.8 (2; 1 row, two rounds of workgroups: 15.5); tile 2048: 40 / 13.0 (1)
//   20,011 x 169, tile 4096: 53 / 15.7 (2; 1 row: 18.9)
//   131,072 x 85, tile 1024: 38 / 24.6 (5); tile 2048: 45 / 24.8 (4); tile 4096: 53 / 26.4 (4)
// and where one round needs more than 16 rows, 16 are the fastest or within 3 %
// (700,001 x 85, tile 2048: 6 / 8 / 12 / 16 rows 100 / 97 / 102 / 98).
// The FOP does not depend on it.
void fit_ftc_items(std::vector<FtcJob>& jobs, uint32_t slots);

// Template spectra (T x S, natural order, complex double) -> kernel layout
// [t][slot][tid], scaled by 1/S (exact).
std::vector<float2> kernel_template_layout(const std::vector<std::complex<double>>& spec, uint32_t n_templates,
                                           uint32_t tile);

// Taps (T x n_taps complex float) -> natural-order spectra of size tile; extent[t]
// receives the non-zero length of each row (at least 1).
std::vector<std::complex<double>> taps_to_spectra(const float* taps_c64, uint32_t n_templates, uint32_t n_taps,
                                                  uint32_t max_taps, uint32_t tile, std::vector<uint32_t>& extent);

// Twiddle tables of the S-point tile transform: w1[k][b] = W_S^(b k), w2[k][d] = W_(S/16)^(d k).
void make_twiddles(uint32_t tile, std::vector<float2>& tw1, std::vector<float2>& tw2);

// The front end's twiddle tables, one after another, for its column (len[0]) and row (len[1]) transforms.  A line
// of L = 16 NT points reads w1 where NT > 1 and w2 where it takes three passes (L > 256); no other table is made,
// and two transforms of one length share theirs.
struct LineTables {
  std::vector<float2> data;
  uint32_t w1[2] = {0, 0}, w2[2] = {0, 0};  // where each begins
};
LineTables line_tables(const uint32_t (&len)[2]);

// Rows per summing workgroup for a launch of one trial.  Short chunks fill the
// chip where a plane is small (a chunk's rows follow one another, and each waits
// for its loads); tall ones re-read fewer sub-harmonic rows and send fewer additions
// to each plane's detection count, which take turns at about 6 ns.  Between, the best
// height grows with the square root of the plane's size.  Measured, us of the kernel
// at 8 planes and 2 / 4 / 8 / 11 rows: 4,999 bins x 33 rows (4 planes; 1 row 4.7)
// 5.7 / 9.0 / 15 / 21; 20,011 x 169 15 / 14 / 23 / 31; 32,768 x 85 12.7 / 10.6 / 18 / 22;
// 100,003 x 85 31 / 22 / 17 / 17; 262,144 x 85 70 / 44 / 33 / 34; 700,001 x 85
// 175 / 105 / 72 / 65; 2^21 x 85 510 / 302 / 200 / 196, and 203 at 15.
// The rule does not look at the number of planes.  Against the fastest of 1, 2, 4, 8,
// 11 and 16 rows on a spectrum with a tone that every plane detects, it is within
// 25 % at 1 and 2 planes and within 10 % at 4 and 8; at 12 and 16 fewer rows would be
// faster: 100,003 x 85 at 4 rows 28 and 33 us against 34 and 44, 2^21 x 85 at 8 rows
// 340 and 439 against 389 and 504.
uint32_t hsum_rows_for(uint32_t n_bins, uint32_t n_rows);

// HSUM workgroup row chunking for a part of n_rows rows (at most `target` rows per workgroup).
void hsum_row_chunks(uint32_t n_rows, uint32_t* rows_per_block, uint32_t* n_row_chunks,
                     uint32_t target = kHsumRowsPerBlock);

}  // namespace fdas
