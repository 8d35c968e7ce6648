// Host-side entry points of the device kernels (implemented in fdas_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fdas_jobs.h"
#include "fdas_select.h"

namespace fdas {

constexpr int kHsumThreads = 256;
constexpr int kHsumBinsPerThread = 8;
constexpr int kHsumBinsPerBlock = kHsumThreads * kHsumBinsPerThread;  // bins one HSUM workgroup covers
// Rows of whole 8-bin groups (part of the rule for the fused kernel).
inline bool hsum_whole_groups(uint32_t n_bins) { return n_bins % kHsumBinsPerThread == 0; }
constexpr uint32_t kHsumRowsPerBlock = 11;  // target rows per HSUM workgroup (bounds the dense-hit tail)
constexpr uint32_t kSelectMaxCap = 8192;  // largest per-plane cap the in-LDS sort handles
constexpr uint32_t kSelectPool = 4096;    // boundary-bin entries resolved exactly in LDS
constexpr uint32_t kSelectSlices = 64;    // workgroups per plane in the histogram / compaction passes

int ftconv_threads(int tile);

// Times of a launch sequence are read on the device: a kernel given a `stamp` has its first workgroup write the
// device's constant-rate clock there (pinned host memory) as it starts.  An event between two kernels is a packet of
// its own, or a signal on the dispatch, that keeps the second kernel waiting for 5 to 9 us: with three events in it a
// launch of 32768 bins took 106 us, with none 88, and 85 with stamps and the spectrum copied by a kernel.

// Workgroups of the FT-convolution kernel that run at once on n_cu CUs, at three
// waves per SIMD: 12 one-wave workgroups per CU for 1024-point tiles, 6 and 3 of two
// and four waves for 2048 and 4096.
inline uint32_t ftconv_slots(uint32_t tile, uint32_t n_cu) { return n_cu * 12u * 1024u / tile; }

// Fused FT convolution over a list of jobs (all with the same tile size).
hipError_t launch_ftconv(int tile, const FtcJob* d_jobs, uint32_t n_jobs, uint32_t n_items, const float2* tw1,
                         const float2* tw2, uint32_t grid, hipStream_t stream, uint64_t* stamp = nullptr);

// Forward transform of every tile of one spectrum, natural bin order (debug / drop-in retrieve_tiles).
hipError_t launch_tiles(int tile, const float2* spectrum, uint32_t n_bins, uint32_t overlap, uint32_t payload,
                        uint32_t n_tiles, const float2* tw1, const float2* tw2, float2* out, hipStream_t stream);

// Harmonic summing + thresholding + compaction into per-plane spill lists.
// All jobs of one launch share n_harmonics; any row lengths go together.
hipError_t launch_hsum(const HsumJob* d_jobs, uint32_t n_jobs, uint32_t n_blocks, uint32_t n_harmonics,
                       hipStream_t stream, uint64_t* stamp = nullptr);

// Per-plane cap (strongest first) and sort by (row, bin): power histogram and
// compaction over the spill lists (kSelectSlices workgroups per plane), then one
// workgroup per plane resolves the boundary bin exactly and sorts.  cap: the
// largest cap of the jobs; ends[n_jobs]: when each plane's lists were complete.
hipError_t launch_select(const SelectJob* d_jobs, uint32_t n_jobs, uint32_t cap, hipStream_t stream,
                         uint64_t* stamp = nullptr, uint64_t* ends = nullptr);

// Harmonic plane HP_k over rows [row_begin, row_begin + n_rows) (debug / parity).
hipError_t launch_hplane(const float* fop, uint32_t n_bins, uint32_t n_templates, uint32_t row_begin,
                         uint32_t n_rows, uint32_t k, float* out, hipStream_t stream);

// Per-block maxima of HP_1 .. HP_H over a part (blocks of 256 bins x 8 rows),
// out[k-1][block] for hmax_blocks(n_bins, n_rows) blocks per plane.
uint32_t hmax_blocks(uint32_t n_bins, uint32_t n_rows);
hipError_t launch_hmax(const float* fop, uint32_t n_bins, uint32_t n_templates, uint32_t row_begin, uint32_t n_rows,
                       uint32_t n_harmonics, float* out, hipStream_t stream);

// The quantile thresholds' order statistics.  launch_quantile_bound sets the
// thresholds of a summing job (and its n_harmonics selection jobs, and thr_out[H])
// to bounds that `want` values of each plane lie above, from its nb block maxima;
// launch_quantile_rank reads the planes' spill lists: out[3H] = detections, value
// bits at descending rank r_lo, at r_hi.
hipError_t launch_quantile_bound(const float* maxima, uint32_t nb, uint32_t want, uint32_t n_harmonics,
                                 HsumJob* d_hsum, SelectJob* d_sel, float* thr_out, hipStream_t stream);
hipError_t launch_quantile_rank(const SelectJob* d_sel, uint32_t n_harmonics, uint32_t r_lo, uint32_t r_hi,
                                uint32_t* out, hipStream_t stream);

// Clears what a summing and selection pass counts in (detections, compact counts, histograms).
hipError_t launch_clear_counters(const SelectJob* d_jobs, uint32_t n_jobs, hipStream_t stream);

hipError_t launch_zero_u32(uint32_t* p, uint32_t n, hipStream_t stream);

// The job descriptors of one trial's launches, taken to the device as the argument
// of a kernel that also clears the counters: one launch in place of
// three copies and a fill.
constexpr uint32_t kPackFtcJobs = 16;
struct JobPack {
  FtcJob ftc[kPackFtcJobs];
  HsumJob hsum;
  SelectJob sel[kMaxHarmonics];
  uint32_t n_ftc = 0, n_sel = 0;  // descriptors to write (the summing job goes with the selection jobs)
};
struct ZeroSpan {
  uint32_t* p = nullptr;
  uint32_t n = 0;
};
// Times that a sequence has not reached are cleared by its first kernel, in the stream's order: the host cannot, while
// an earlier sequence may still write them.
struct StampSpan {
  uint64_t* p = nullptr;
  uint32_t n = 0;  // at most a workgroup of put_jobs, copy_spectrum or stamp_kernel (64)
};
// What put_jobs does with a sequence's times: *keep_to = *keep_from, then the clearing, then the stamps.
struct StampOps {
  uint64_t* stamp = nullptr;
  uint64_t* stamp2 = nullptr;
  StampSpan clear;
  const uint64_t* keep_from = nullptr;
  uint64_t* keep_to = nullptr;
};
hipError_t launch_put_jobs(const JobPack& pack, FtcJob* d_ftc, HsumJob* d_hsum, SelectJob* d_sel, ZeroSpan zero,
                           hipStream_t stream, const StampOps& times = StampOps{});

// n spectrum bins from device or pinned host memory (8-byte aligned); `end`: the last workgroup's end.
hipError_t launch_copy_spectrum(const float2* src, float2* dst, uint32_t n, hipStream_t stream, uint64_t* stamp,
                                uint64_t* end, StampSpan clear);

// A stamp where no kernel of the sequence starts.
hipError_t launch_stamp(hipStream_t stream, uint64_t* stamp, uint64_t* stamp2 = nullptr, StampSpan clear = StampSpan{});

// One launch running both the FT convolution of ftc_jobs (1024-point tiles)
// and the harmonic summing of hsum_jobs (n_harmonics planes) over a FOP written
// by an earlier launch; workgroups of the two kinds are interleaved.
// fused_supported tells which shapes it covers (whole_groups: every row length
// is a multiple of 8).
bool fused_supported(uint32_t tile, uint32_t n_harmonics, bool whole_groups);
hipError_t launch_fused(const FtcJob* ftc_jobs, uint32_t n_ftc_jobs, uint32_t n_items, const float2* tw1,
                        const float2* tw2, const HsumJob* hsum_jobs, uint32_t n_hsum_jobs, uint32_t n_blocks,
                        uint32_t n_harmonics, hipStream_t stream);

}  // namespace fdas
