// Device kernels of the FDAS hot path for CDNA4 (gfx950).
//
//  ftconv_kernel  fused overlap-save FT convolution: tile load -> forward FFT
//                 -> x template spectrum -> inverse FFT -> discard overlap -> |x|^2
//                 (reference: tile_input.cl.mako, fft.cl.mako, mux_and_mult.cl.mako,
//                  square_and_discard.cl.mako; oracle ft_conv.py:158-207)
//  hsum_kernel    harmonic summing + per-plane strict thresholding + compaction
//                 (reference: hms_baseline.cl.mako:55-71, detect.cl.mako:81-104,
//                  hsum.py:91-151)
//  select_kernel  per-plane cap (strongest first) and (row, bin) ordering of the
//                 detections; replaces the reference's overwrite-oldest ring
//                 (detect.cl.mako:106-115) with a deterministic rule.
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "fdas_kernels.h"
#include "fft_tile.h"

namespace fdas {

// ---------------------------------------------------------------------------
// FT convolution
// ---------------------------------------------------------------------------

__device__ __forceinline__ void put_stamp(uint64_t* stamp) {
  if (stamp && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *stamp = wall_clock64();
}

__device__ __forceinline__ void clear_stamps(StampSpan s) {
  if (blockIdx.x == 0 && threadIdx.x < s.n) s.p[threadIdx.x] = 0;
}

__device__ __forceinline__ uint32_t find_job_ftc(const FtcJob* __restrict__ jobs, uint32_t n_jobs, uint32_t item) {
  uint32_t lo = 0, hi = n_jobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (jobs[mid].item_begin <= item) lo = mid; else hi = mid;
  }
  return lo;
}

// 2048- and 4096-point tiles, S / 16 threads (2 and 4 waves) per workgroup.
//
// Bound by VALU issue and, for a launch of a round or two, by latency.  Held to 168
// registers (three waves per SIMD): F2 twiddles in LDS, one exchange buffer, template
// spectra loaded when they are used.  With everything in registers, two buffers and
// the template prefetched one row ahead (232 / 221 VGPRs, two waves) a trial of
// 85 templates took, 2048-point tiles: 50 us at 2^18 bins, 114 at 700,001, 350 at
// 2^21, against 46, 99 and 336; 4096-point tiles at 2^21: 373 against 338.  The FMA
// forms are spelled out to give the FOP that kernel gave, bit for bit.
template <int S>
__global__ __launch_bounds__(S / 16) __attribute__((amdgpu_waves_per_eu(3, 3))) void ftconv_kernel(
    const FtcJob* __restrict__ jobs, uint32_t n_jobs, uint32_t n_items, const float2* __restrict__ tw1,
    const float2* __restrict__ tw2, uint64_t* stamp) {
  put_stamp(stamp);
  using F = TileFFTLean<S>;
  constexpr int NT = F::NT;
  __shared__ float2 la[F::LDS_ELEMS];
  __shared__ float2 w2[F::W2_ELEMS];
  const int tid = threadIdx.x;
  F fft;
  fft.load_twiddles(tw1, tw2, w2, tid);

  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const FtcJob* job = jobs + find_job_ftc(jobs, n_jobs, item);
    const uint32_t n_bins = job->n_bins;
    const uint32_t overlap = job->overlap;
    const uint32_t payload = job->payload;
    const uint32_t local = item - job->item_begin;
    const uint32_t chunk = local / job->n_tiles;  // consecutive items share a template chunk
    const uint32_t tile = local - chunk * job->n_tiles;
    const float2* __restrict__ x = static_cast<const float2*>(job->spectrum);

    __syncthreads();  // previous item's LDS readers are done

    float2 xf[16];
    const int base = int(tile * payload) - int(overlap);
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int idx = base + NT * a + tid;
      xf[a] = make_float2(0.f, 0.f);
      if (idx >= 0 && idx < int(n_bins)) xf[a] = gld2(x, size_t(idx));
    }

    const uint32_t r_begin = job->row_begin + chunk * job->rows_per_item;
    uint32_t r_end = r_begin + job->rows_per_item;
    const uint32_t r_stop = job->row_begin + job->n_rows;
    if (r_end > r_stop) r_end = r_stop;
    const float2* __restrict__ hbase = static_cast<const float2*>(job->hperm);
    const uint32_t out0 = tile * payload;  // FOP bin of tile sample s = overlap

    fft.forward(xf, la, tid);
    for (uint32_t r = r_begin; r < r_end; ++r) {
      float2 v[16];
#pragma unroll
      for (int s = 0; s < 16; ++s) v[s] = cmul_f0(xf[s], gld2(hbase + size_t(r) * S + tid, size_t(s * NT)));
      fft.inverse(v, la, tid);
      // Slot a of this thread is FOP bin out0 + NT*a + tid - overlap: one base
      // address per row and a constant offset per slot (the store's immediate).
      float* __restrict__ out = job->fop + size_t(r) * n_bins + (ptrdiff_t(out0) + tid - ptrdiff_t(overlap));
#pragma unroll
      for (int a = 0; a < 16; ++a) {
        const uint32_t s = uint32_t(NT * a + tid);
        if (s >= overlap) {
          const uint32_t f = out0 + s - overlap;
          if (f < n_bins) gst_stream(out, size_t(NT * a), v[a].x * v[a].x + v[a].y * v[a].y);
        }
      }
    }
  }
}

// 1024-point work items for four-wave workgroups (the fused launch below):
// wave 0 loads the tile and forward-transforms it into LDS (xs); then every
// wave convolves its share of the item's template rows (rows w, w + 4, ...),
// each row reading the tile spectrum back from LDS, so the workgroup runs at
// three waves per SIMD.
constexpr int kFtc1kWaves = 4;

// LDS of one 1024-point work item, carved from a caller's buffer.
struct Ftc1kLds {
  float2 xs[16 * WaveFFT1k<true>::NT];                   // the tile's spectrum, slot-major
  float2 lbuf[kFtc1kWaves][WaveFFT1k<true>::LDS_ELEMS];  // each wave's exchange buffer
  float2 w2s[64];                                  // W_64^(d * kc), the F2 twiddles
};

// One work item (tile, chunk of template rows) of a 1024-point job list.
// `fft` holds this thread's twiddles; `first` is true for the workgroup's
// first item (wave 0 has just filled w2s: the first barrier publishes it).
__device__ __forceinline__ void ftc1k_item(Ftc1kLds& L, const WaveFFT1k<true>& fft,
                                           const FtcJob* __restrict__ jobs, uint32_t n_jobs, uint32_t item) {
  using F = WaveFFT1k<true>;
  constexpr int NT = F::NT;
  constexpr int S = F::S;
  const int lane = int(threadIdx.x) & 63;
  const uint32_t wave = threadIdx.x >> 6;
  float2* __restrict__ lb = L.lbuf[wave];
  const FtcJob* job = jobs + find_job_ftc(jobs, n_jobs, item);
  const uint32_t n_bins = job->n_bins;
  const uint32_t overlap = job->overlap;
  const uint32_t payload = job->payload;
  const uint32_t local = item - job->item_begin;
  const uint32_t chunk = local / job->n_tiles;  // consecutive items share a template chunk
  const uint32_t tile = local - chunk * job->n_tiles;
  const uint32_t r_begin = job->row_begin + chunk * job->rows_per_item;
  uint32_t r_end = r_begin + job->rows_per_item;
  const uint32_t r_stop = job->row_begin + job->n_rows;
  if (r_end > r_stop) r_end = r_stop;
  const float2* __restrict__ hbase = static_cast<const float2*>(job->hperm);
  const uint32_t out0 = tile * payload;  // FOP bin of tile sample s = overlap

  // This wave's first template row is loaded before the forward transform,
  // every next one as soon as the current one has been used.
  uint32_t r = r_begin + wave;
  float2 hn[16];
  {
    const float2* __restrict__ h = hbase + size_t(min(r, r_end - 1)) * S + lane;
#pragma unroll
    for (int s = 0; s < 16; ++s) hn[s] = gld2(h, size_t(s * NT));
  }

  __syncthreads();  // every wave has finished reading the previous item's spectrum
  if (wave == 0) {
    const float2* __restrict__ x = static_cast<const float2*>(job->spectrum);
    float2 v[16];
    const int base = int(tile * payload) - int(overlap);
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int idx = base + NT * a + lane;
      v[a] = make_float2(0.f, 0.f);
      if (idx >= 0 && idx < int(n_bins)) v[a] = gld2(x, size_t(idx));
    }
    fft.forward(v, lb, lane);
#pragma unroll
    for (int s = 0; s < 16; ++s) L.xs[s * NT + lane] = v[s];
  }
  __syncthreads();

  for (; r < r_end; r += kFtc1kWaves) {
    float2 v[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) v[s] = cmul(L.xs[s * NT + lane], hn[s]);
    {
      const float2* __restrict__ h = hbase + size_t(min(r + kFtc1kWaves, r_end - 1)) * S + lane;
#pragma unroll
      for (int s = 0; s < 16; ++s) hn[s] = gld2(h, size_t(s * NT));
    }
    fft.inverse(v, lb, lane);
    float* __restrict__ out = job->fop + size_t(r) * n_bins + (ptrdiff_t(out0) + lane - ptrdiff_t(overlap));
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const uint32_t s = uint32_t(NT * a + lane);
      if (s >= overlap) {
        const uint32_t f = out0 + s - overlap;
        if (f < n_bins) gst_stream(out, size_t(NT * a), v[a].x * v[a].x + v[a].y * v[a].y);
      }
    }
  }
}

// 1024-point tiles, one wave per workgroup.  The tile's spectrum and the
// twiddles stay in registers; the F2 <-> F3 exchange is a pair of permlane
// swaps and only the F1 <-> F2 exchange goes through LDS (8.3 KB per
// workgroup).  164 VGPRs: three waves per SIMD.
__global__ __launch_bounds__(64) void ftconv1w_kernel(const FtcJob* __restrict__ jobs, uint32_t n_jobs,
                                                      uint32_t n_items, const float2* __restrict__ tw1,
                                                      const float2* __restrict__ tw2, uint64_t* stamp) {
  put_stamp(stamp);
  using F = WaveFFT1kLean;
  constexpr int NT = F::NT;
  constexpr int S = F::S;
  __shared__ float2 lb[F::LDS_ELEMS];
  const int lane = threadIdx.x;
  F fft;
  fft.load_twiddles(tw1, tw2, lane);

  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const FtcJob* job = jobs + find_job_ftc(jobs, n_jobs, item);
    const uint32_t n_bins = job->n_bins;
    const uint32_t overlap = job->overlap;
    const uint32_t payload = job->payload;
    const uint32_t local = item - job->item_begin;
    const uint32_t chunk = local / job->n_tiles;
    const uint32_t tile = local - chunk * job->n_tiles;
    const float2* __restrict__ x = static_cast<const float2*>(job->spectrum);
    const uint32_t r_begin = job->row_begin + chunk * job->rows_per_item;
    uint32_t r_end = r_begin + job->rows_per_item;
    const uint32_t r_stop = job->row_begin + job->n_rows;
    if (r_end > r_stop) r_end = r_stop;
    const float2* __restrict__ hbase = static_cast<const float2*>(job->hperm);
    const uint32_t out0 = tile * payload;

    float2 xf[16];
    const int base = int(tile * payload) - int(overlap);
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const int idx = base + NT * a + lane;
      xf[a] = make_float2(0.f, 0.f);
      if (idx >= 0 && idx < int(n_bins)) xf[a] = gld2(x, size_t(idx));
    }
    fft.forward(xf, lb, lane);
    for (uint32_t r = r_begin; r < r_end; ++r) {
      // The template spectrum is not prefetched: at three waves per SIMD the
      // other waves' transforms cover the load.
      float2 v[16];
#pragma unroll
      for (int s = 0; s < 16; ++s) v[s] = cmul(xf[s], gld2(hbase + size_t(r) * S + lane, size_t(s * NT)));
      fft.inverse(v, lb, lane);
      float* __restrict__ out = job->fop + size_t(r) * n_bins + (ptrdiff_t(out0) + lane - ptrdiff_t(overlap));
#pragma unroll
      for (int a = 0; a < 16; ++a) {
        const uint32_t s = uint32_t(NT * a + lane);
        if (s >= overlap) {
          const uint32_t f = out0 + s - overlap;
          if (f < n_bins) gst_stream(out, size_t(NT * a), v[a].x * v[a].x + v[a].y * v[a].y);
        }
      }
    }
  }
}

template <int S>
__global__ __launch_bounds__(S / 16) void tiles_kernel(const float2* __restrict__ x, uint32_t n_bins,
                                                       uint32_t overlap, uint32_t payload,
                                                       const float2* __restrict__ tw1,
                                                       const float2* __restrict__ tw2, float2* __restrict__ out) {
  using F = TileFFT<S>;
  constexpr int NT = F::NT;
  __shared__ float2 la[F::LDS_ELEMS];
  const int tid = threadIdx.x;
  F fft;
  fft.load_twiddles(tw1, tw2, tid);
  const uint32_t tile = blockIdx.x;
  const int base = int(tile * payload) - int(overlap);
  float2 v[16];
#pragma unroll
  for (int a = 0; a < 16; ++a) {
    const int idx = base + NT * a + tid;
    v[a] = (idx >= 0 && idx < int(n_bins)) ? x[idx] : make_float2(0.f, 0.f);
  }
  fft.forward(v, la, tid);
  float2* __restrict__ o = out + size_t(tile) * S;
#pragma unroll
  for (int s = 0; s < 16; ++s) o[F::slot_bin(tid, s)] = v[s];
}

int ftconv_threads(int tile) { return tile == 1024 ? 64 : tile / 16; }

hipError_t launch_ftconv(int tile, const FtcJob* d_jobs, uint32_t n_jobs, uint32_t n_items, const float2* tw1,
                         const float2* tw2, uint32_t grid, hipStream_t stream, uint64_t* stamp) {
  if (n_items == 0) return hipSuccess;
  if (grid == 0 || grid > n_items) grid = n_items;
  switch (tile) {
    case 1024: ftconv1w_kernel<<<grid, 64, 0, stream>>>(d_jobs, n_jobs, n_items, tw1, tw2, stamp); break;
    case 2048: ftconv_kernel<2048><<<grid, 128, 0, stream>>>(d_jobs, n_jobs, n_items, tw1, tw2, stamp); break;
    case 4096: ftconv_kernel<4096><<<grid, 256, 0, stream>>>(d_jobs, n_jobs, n_items, tw1, tw2, stamp); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_tiles(int tile, const float2* spectrum, uint32_t n_bins, uint32_t overlap, uint32_t payload,
                        uint32_t n_tiles, const float2* tw1, const float2* tw2, float2* out, hipStream_t stream) {
  if (n_tiles == 0) return hipSuccess;
  switch (tile) {
    case 1024: hipLaunchKernelGGL(tiles_kernel<1024>, dim3(n_tiles), dim3(64), 0, stream, spectrum, n_bins, overlap, payload, tw1, tw2, out); break;
    case 2048: hipLaunchKernelGGL(tiles_kernel<2048>, dim3(n_tiles), dim3(128), 0, stream, spectrum, n_bins, overlap, payload, tw1, tw2, out); break;
    case 4096: hipLaunchKernelGGL(tiles_kernel<4096>, dim3(n_tiles), dim3(256), 0, stream, spectrum, n_bins, overlap, payload, tw1, tw2, out); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Harmonic summing
// ---------------------------------------------------------------------------

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}

// Exclusive prefix sum over the wave of a per-lane count v < 16, bit-sliced:
// one ballot per bit.  `total` receives the wave's sum (wave-uniform).
__device__ __forceinline__ uint32_t wave_prefix_small(uint32_t v, uint32_t& total) {
  uint32_t excl = 0;
  total = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint64_t m = __ballot((v >> j) & 1u);
    excl += lanes_below(m) << j;
    total += uint32_t(__builtin_popcountll(m)) << j;
  }
  return excl;
}

// Per-wave detection staging.  A lane with a hit stages its whole group, 8 sums
// and their first key, in one slot of its wave's list for the plane; the bins
// that pass are picked out when the list is flushed, by 8 lanes per group.  So a
// hit costs the row loop one ballot and three LDS writes: picking the bins there
// (compares, a prefix sum and a store per bin, inlined for each plane and
// register buffer) took about 170 instructions, and two rows in three have a
// wave with a hit at six-sigma thresholds.  8 trials of 2^21 bins x 85 rows x 8
// planes 1.645 -> 1.617 ms (memory bound), 2^20 x 85 x 16 1.54 -> 1.48.
template <int H>
struct HsumStage {
  static constexpr uint32_t kGroups = H <= 8 ? 24 : 12;  // 27.8 KB at 8 planes, 27.9 at 16: 5 workgroups per CU
  float sum[kHsumThreads / 64][H][kGroups][kHsumBinsPerThread];
  uint32_t key[kHsumThreads / 64][H][kGroups];  // row << kKeyBinBits | f0
  uint32_t n[H][kHsumThreads / 64];             // groups of each wave, at the end
};

// One bin of each of 8 staged groups, first, first + 1, ...: this lane's value and key,
// and whether it is a hit of the plane.
template <class Stage>
__device__ __forceinline__ bool staged_bin(const Stage& st, uint32_t wave, uint32_t p, uint32_t first, uint32_t n,
                                           float thr, uint32_t n_bins, float* v, uint32_t* key) {
  const uint32_t lane = lane_id(), g = first + lane / 8u, b = lane % 8u;
  if (g >= n) return false;
  *v = st.sum[wave][p][g][b];
  *key = st.key[wave][p][g] + b;
  return *v > thr && (*key & ((1u << kKeyBinBits) - 1u)) < n_bins;
}

__device__ __forceinline__ void spill_hit(const HsumJob& job, uint32_t p, uint32_t slot, uint32_t key, float v) {
  if (slot >= job.spill_cap) return;  // counted, not kept
  gst(job.spill_key, size_t(p) * job.spill_cap + slot, key);
  gst(job.spill_pwr, size_t(p) * job.spill_cap + slot, v);
}

// Writes the hits of the wave's n staged groups of plane p to the global spill
// list, with one global atomic.
template <class Stage>
__device__ __forceinline__ void wave_flush(Stage& st, const HsumJob& job, uint32_t wave, uint32_t p, uint32_t n,
                                           float thr) {
  constexpr int kSteps = int((Stage::kGroups + 7) / 8);
  wave_lds_order();
  float v[kSteps];
  uint32_t key[kSteps], slot[kSteps], total = 0;
  bool hit[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    hit[s] = staged_bin(st, wave, p, uint32_t(8 * s), n, thr, job.n_bins, &v[s], &key[s]);
    const uint64_t m = __ballot(hit[s]);
    slot[s] = total + lanes_below(m);
    total += uint32_t(__builtin_popcountll(m));
  }
  wave_lds_order();  // the stage is rewritten next
  if (total == 0) return;
  uint32_t base = 0;
  if (lane_id() == 0) base = gatomic_add(job.counts + size_t(p) * kPlaneCounters, total);
  base = __shfl(base, 0);
#pragma unroll
  for (int s = 0; s < kSteps; ++s)
    if (hit[s]) spill_hit(job, p, base + slot[s], key[s], v[s]);
}

__device__ __forceinline__ uint32_t find_job_hsum(const HsumJob* __restrict__ jobs, uint32_t n_jobs, uint32_t blk) {
  uint32_t lo = 0, hi = n_jobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (jobs[mid].block_begin <= blk) lo = mid; else hi = mid;
  }
  return lo;
}

// A thread sums 8 consecutive bins f0 .. f0+7 of a row, f0 a multiple of 8.
// For harmonic k their sub-harmonic bins (f0 + b) / k are the hsum_span(k)
// consecutive bins from f0 / k: f0 mod k is a multiple of g = gcd(8, k), at
// most k - g, so the last one is at most (k - g + 7) / k bins further on.
__host__ __device__ constexpr int hsum_gcd8(int k) { return (k % 8 == 0) ? 8 : (k % 4 == 0) ? 4 : (k % 2 == 0) ? 2 : 1; }
__host__ __device__ constexpr int hsum_span(int k) { return 1 + (k - hsum_gcd8(k) + 7) / k; }
constexpr int kHsumMaxSpan = 4;  // hsum_span(2) = hsum_span(3) = 4 is the largest
static_assert(kHsumBinsPerThread == 8, "the sub-harmonic spans assume 8 bins per thread");

// Every FOP value one thread needs for one row: its 8 own bins and, for each
// harmonic k >= 2, the hsum_span(k) sub-harmonic bins of row trunc(t / k).
template <int H>
struct RowLoads {
  float m[kHsumBinsPerThread];
  float s[H][kHsumMaxSpan];
};

// Branch-free: H is a compile-time constant and every index is in range, so
// the compiler can count the loads in flight exactly (a load issued under a
// condition makes it drain every outstanding load at the next use).
//
// n_bins >= 8 may be any length: the loads need dword alignment only.  Bound by
// HBM traffic as long as they stay wide: 16-byte loads of the own bins and of
// the k = 2, 3 spans, narrower ones that the compiler merges for the rest, 9 per
// row at H = 8.  With one dword load per value and a clamp on each (135 VGPRs,
// 3 waves per SIMD) rows of odd length took 124 us per 700,001 bins x 43 rows,
// against 57 us this way, and since a launch ran in one form for all its jobs,
// one odd-length trial among five took the launch from 0.98 to 3.29 ms.
//
// A thread whose group of 8 crosses the end of its row reads on into the next
// row (live_bits masks what it finds there); the plane's last row has no next
// one, so hsum_block sums that row of the last wave bin by bin.
//
// For n_bins >= 8 a sub-harmonic span ends at (n_bins - 1) / 2 + 3 <= n_bins - 1
// at most.
template <int H>
__device__ __forceinline__ void hsum_load_row(RowLoads<H>& L, const float* __restrict__ fop, uint32_t n_bins, int c,
                                              uint32_t r, uint32_t f0) {
  const float* __restrict__ row = fop + size_t(r) * n_bins;
  const fdas_vf4u q0 = gld4u(row, f0);
  const fdas_vf4u q1 = gld4u(row, f0 + 4);
  L.m[0] = q0.x; L.m[1] = q0.y; L.m[2] = q0.z; L.m[3] = q0.w;
  L.m[4] = q1.x; L.m[5] = q1.y; L.m[6] = q1.z; L.m[7] = q1.w;
  const int t = int(r) - c;
#pragma unroll
  for (int k = 2; k <= H; ++k) {
    const float* __restrict__ srow = fop + size_t(c + t / k) * n_bins;
    const uint32_t s0 = f0 / uint32_t(k);
    if (k == 2) {
      const fdas_vf4u q = gld4u(srow, s0);
      L.s[k - 1][0] = q.x; L.s[k - 1][1] = q.y; L.s[k - 1][2] = q.z; L.s[k - 1][3] = q.w;
    } else if (k == 4) {
      const fdas_vf2u q = gld2u(srow, s0);
      L.s[k - 1][0] = q.x; L.s[k - 1][1] = q.y;
    } else {
#pragma unroll
      for (int j = 0; j < hsum_span(k); ++j) L.s[k - 1][j] = gld(srow, s0 + uint32_t(j));
    }
  }
}

// Bin b of the thread takes sub-harmonic value (f0 mod k + b) / k of its span:
// b / k when f0 mod k < k (b / k + 1) - b, else the next one.  rk[k-1] = f0 mod k
// is a multiple of g = gcd(8, k), so the edge may be rounded up to one: that
// drops the selects no residue reaches, and bins share their compares (35 in
// place of 49 for k = 9 .. 15; 1.61 -> 1.54 ms per 8 trials of 2^20 bins x 85 rows
// x 16 planes, no change at 8 planes).
template <int K>
__device__ __forceinline__ float hsum_sub(const float (&s)[kHsumMaxSpan], uint32_t rk, int b) {
  const int lo = b / K, g = hsum_gcd8(K);
  const int edge = (K * (lo + 1) - b + g - 1) / g * g;  // f0 mod k at which bin b moves to the next value
  if (edge > K - g) return s[lo];  // no f0 mod k reaches it
  return rk >= uint32_t(edge) ? s[lo + 1] : s[lo];
}

template <int H, int K>
__device__ __forceinline__ void hsum_add(float (&hp)[kHsumBinsPerThread], const RowLoads<H>& L, uint32_t rk) {
#pragma unroll
  for (int b = 0; b < kHsumBinsPerThread; ++b) hp[b] += hsum_sub<K>(L.s[K - 1], rk, b);
}

template <int H, int K = 2>
__device__ __forceinline__ void hsum_add_k(int k, float (&hp)[kHsumBinsPerThread], const RowLoads<H>& L,
                                           const uint32_t (&rk)[H]) {
  if constexpr (K <= H) {
    if (k == K) hsum_add<H, K>(hp, L, rk[K - 1]);
    else hsum_add_k<H, K + 1>(k, hp, L, rk);
  }
}

// Key of the per-plane group test: a value v > thr implies
// float_as_int(v) >= group_key(thr) for every v and thr (a non-negative thr
// orders like its bit pattern against any v above it; a negative one admits
// everything), so the test below only ever lets through a superset of the
// bins the exact float compare accepts.
__device__ __forceinline__ int group_key(float thr) { return thr < 0.f ? INT_MIN : __float_as_int(thr); }

// Largest bit pattern of the 8 sums as signed integers: three max3 and one max,
// with no NaN canonicalisation of the operands (which fmaxf would need).
__device__ __forceinline__ int group_max(const float (&hp)[kHsumBinsPerThread]) {
  const int a = max(max(__float_as_int(hp[0]), __float_as_int(hp[1])), __float_as_int(hp[2]));
  const int b = max(max(__float_as_int(hp[3]), __float_as_int(hp[4])), __float_as_int(hp[5]));
  return max(max(a, b), max(__float_as_int(hp[6]), __float_as_int(hp[7])));
}

// One test per plane for the common case: the group key of the 8 sums against
// the plane's; only a wave with a candidate looks at the bins one by one with
// the exact float compare.  The thresholds are wave-uniform; `live_lanes`
// holds the lanes with at least one bin in range (per-bin range checks are in
// `live_bits`, bit b for bin b).
template <int H, class Stage>
__device__ __forceinline__ void hsum_row(Stage& st, const HsumJob& job, const RowLoads<H>& L, uint32_t r,
                                         uint32_t f0, const uint32_t (&rk)[H], const float (&thr)[H],
                                         const int (&thr_key)[H], uint64_t live_lanes, uint32_t live_bits,
                                         uint32_t (&wn)[H], uint32_t wave) {
  float hp[kHsumBinsPerThread];
#pragma unroll
  for (int b = 0; b < kHsumBinsPerThread; ++b) hp[b] = L.m[b];
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    if (k > 1) hsum_add_k<H>(k, hp, L, rk);
    const uint64_t groups = __ballot(group_max(hp) >= thr_key[k - 1]) & live_lanes;
    if (groups == 0) continue;
    const uint32_t n_groups = uint32_t(__builtin_popcountll(groups));
    if (wn[k - 1] + n_groups > Stage::kGroups) {
      wave_flush(st, job, wave, uint32_t(k - 1), wn[k - 1], thr[k - 1]);
      wn[k - 1] = 0;
    }
    if (n_groups > Stage::kGroups) {
      // more than the stage holds (a strong signal, a low threshold): straight to the spill list,
      // the wave's hits in lane order, each lane's in bin order
      uint32_t bits = 0;
#pragma unroll
      for (int b = 0; b < kHsumBinsPerThread; ++b) bits |= (hp[b] > thr[k - 1]) ? (1u << b) : 0u;
      bits &= live_bits;
      uint32_t total;
      const uint32_t pos = wave_prefix_small(uint32_t(__builtin_popcount(bits)), total);
      uint32_t g = 0;
      if (lane_id() == 0) g = gatomic_add(job.counts + size_t((k - 1)) * kPlaneCounters, total);
      g = __shfl(g, 0) + pos;
#pragma unroll
      for (int b = 0; b < kHsumBinsPerThread; ++b) {
        if ((bits >> b) & 1u) {
          spill_hit(job, uint32_t(k - 1), g, (r << kKeyBinBits) | (f0 + uint32_t(b)), hp[b]);
          ++g;
        }
      }
    } else {
      if ((groups >> lane_id()) & 1u) {
        const uint32_t slot = wn[k - 1] + lanes_below(groups);
        float* __restrict__ to = st.sum[wave][k - 1][slot];
#pragma unroll
        for (int b = 0; b < kHsumBinsPerThread; ++b) to[b] = hp[b];
        st.key[wave][k - 1][slot] = (r << kKeyBinBits) | f0;
      }
      wn[k - 1] += n_groups;
    }
  }
}

// Writes what the workgroup has staged to the spill lists, with one global atomic per plane.  Many launches are one
// round of workgroups and end with this, so its latency counts.  A wave takes whole planes, the groups of all four
// waves' lists in steps of 8: the waves share a strong signal that one of them has staged, and each wave reserves
// places for its planes with one instruction and needs no second barrier.  (Each wave counting its own lists of all
// planes, one after another, then workgroup totals: 4,999 bins x 33 rows x 8 planes with two tones 10 us against 6.8,
// 32,768 x 85 14.7 against 12.8 at 2 rows a workgroup, 2^20 x 85 x 16 planes 169 against 161.)
template <int H>
__device__ __forceinline__ void flush_rest(HsumStage<H>& st, const HsumJob& job, const uint32_t (&wn)[H]) {
  constexpr uint32_t kWaves = kHsumThreads / 64, kPlanes = (uint32_t(H) + kWaves - 1) / kWaves;  // planes of a wave
  const uint32_t lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t mine = 0;
#pragma unroll
  for (int k = 0; k < H; ++k)
    if (lane == uint32_t(k)) mine = wn[k];
  if (lane < uint32_t(H)) st.n[lane][wave] = mine;
  __syncthreads();
  uint32_t at[kPlanes][kWaves], n[kPlanes];  // where each wave's groups begin in the plane's list; its length
#pragma unroll
  for (uint32_t i = 0; i < kPlanes; ++i) {
    const uint32_t p = wave + i * kWaves;
    n[i] = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
      at[i][w] = n[i];
      n[i] += p < uint32_t(H) ? __builtin_amdgcn_readfirstlane(st.n[p][w]) : 0u;
    }
  }
  // This lane's bin of the groups first .. first + 7 of the wave's plane i.
  auto staged = [&](uint32_t i, uint32_t first, float* v, uint32_t* key) {
    const uint32_t p = wave + i * kWaves, g = first + lane / 8u;
    uint32_t w = 0, begin = 0;
#pragma unroll
    for (uint32_t x = 1; x < kWaves; ++x) {
      if (g < at[i][x]) continue;
      w = x;
      begin = at[i][x];
    }
    if (g >= n[i]) return false;
    *v = st.sum[w][p][g - begin][lane % 8u];
    *key = st.key[w][p][g - begin] + lane % 8u;
    return *v > job.thr[p] && (*key & ((1u << kKeyBinBits) - 1u)) < job.n_bins;
  };
  uint32_t key[kPlanes], hits = 0, x;
  float v[kPlanes], y;
  uint64_t m[kPlanes];  // hits of the first 8 groups, most often all of them
#pragma unroll
  for (uint32_t i = 0; i < kPlanes; ++i) m[i] = __ballot(staged(i, 0, &v[i], &key[i]));
#pragma unroll
  for (uint32_t i = 0; i < kPlanes; ++i) {
    uint32_t total = uint32_t(__builtin_popcountll(m[i]));
    for (uint32_t first = 8; first < n[i]; first += 8)
      total += uint32_t(__builtin_popcountll(__ballot(staged(i, first, &y, &x))));
    if (lane == i) hits = total;
  }
  uint32_t place = 0;
  if (hits) place = gatomic_add(job.counts + size_t(wave + lane * kWaves) * kPlaneCounters, hits);
#pragma unroll
  for (uint32_t i = 0; i < kPlanes; ++i) {
    const uint32_t p = wave + i * kWaves;
    uint32_t to = uint32_t(__builtin_amdgcn_readlane(int(place), int(i)));
    if ((m[i] >> lane) & 1u) spill_hit(job, p, to + lanes_below(m[i]), key[i], v[i]);
    to += uint32_t(__builtin_popcountll(m[i]));
    for (uint32_t first = 8; first < n[i]; first += 8) {
      const bool hit = staged(i, first, &y, &x);
      const uint64_t mask = __ballot(hit);
      if (hit) spill_hit(job, p, to + lanes_below(mask), x, y);
      to += uint32_t(__builtin_popcountll(mask));
    }
  }
}

// One bin of one row, every hit placed by its own atomic: the bins that the
// 16-byte loads cannot cover (below).
template <int H>
__device__ __forceinline__ void hsum_one_bin(const HsumJob& job, uint32_t r, uint32_t f) {
  const int c = int(job.n_templates / 2), t = int(r) - c;
  float v[H];
#pragma unroll
  for (int k = 1; k <= H; ++k) v[k - 1] = gld(job.fop, size_t(c + t / k) * job.n_bins + f / uint32_t(k));
  float hp = v[0];
#pragma unroll
  for (int k = 1; k <= H; ++k) {
    if (k > 1) hp += v[k - 1];
    if (!(hp > job.thr[k - 1])) continue;
    const uint32_t g = gatomic_add(job.counts + size_t((k - 1)) * kPlaneCounters, 1u);
    if (g >= job.spill_cap) continue;
    gst(job.spill_key, size_t(k - 1) * job.spill_cap + g, (r << kKeyBinBits) | f);
    gst(job.spill_pwr, size_t(k - 1) * job.spill_cap + g, hp);
  }
}

// HP_1 = FOP, HP_k = HP_{k-1} + FOP[trunc(t/k)][f/k] in FP32, in k order (hsum.py:93-120);
// strict HP_k > thr_k (detect.cl.mako:81-83).  One workgroup covers 2048 bins
// of a chunk of rows of its part, each thread 8 consecutive bins.  Rows are
// processed in pairs with two register buffers: the loads of row r+1 are in
// flight while row r is summed and thresholded.
template <int H>
__device__ __forceinline__ void hsum_block(HsumStage<H>& st, const HsumJob* __restrict__ jobs, uint32_t n_jobs,
                                           uint32_t blk) {
  const HsumJob& job = jobs[find_job_hsum(jobs, n_jobs, blk)];
  const int tid = threadIdx.x;
  const uint32_t wave = uint32_t(tid) >> 6;

  const uint32_t n_bins = job.n_bins;
  const int c = int(job.n_templates / 2);
  const float* __restrict__ fop = job.fop;
  const uint32_t local = blk - job.block_begin;
  const uint32_t chunk = local % job.n_row_chunks;  // row chunks of one bin block run side by side
  const uint32_t block_f0 = (local / job.n_row_chunks) * uint32_t(kHsumBinsPerBlock);
  const uint32_t f0 = block_f0 + uint32_t(tid * kHsumBinsPerThread);
  const uint32_t r_begin = job.row_begin + chunk * job.rows_per_block;
  const uint32_t r_last = min(r_begin + job.rows_per_block, job.row_begin + job.n_rows) - 1;
  if (n_bins < uint32_t(kHsumBinsPerThread)) {  // rows shorter than one thread's bins
    if (uint32_t(tid) < n_bins)
      for (uint32_t r = r_begin; r <= r_last; ++r) hsum_one_bin<H>(job, r, uint32_t(tid));
    return;
  }
  // The wave that ends in a partial group leaves the plane's last row to the
  // whole workgroup, bin by bin (2 bins per thread).
  constexpr uint32_t kWaveBins = 64u * kHsumBinsPerThread;
  const uint32_t tail_f0 = (n_bins - 1u) / kWaveBins * kWaveBins;
  const bool apart = n_bins % 8u != 0 && r_last + 1u == job.n_templates && tail_f0 - block_f0 < uint32_t(kHsumBinsPerBlock);
  if (apart) {
    for (uint32_t f = tail_f0 + uint32_t(tid); f < min(tail_f0 + kWaveBins, n_bins); f += kHsumThreads)
      hsum_one_bin<H>(job, r_last, f);
  }
  // Threads past the end read (and discard) the row's last group of 8.
  const uint32_t fl = min(f0, (n_bins - 1u) & ~7u);
  float thr[H];
  int thr_key[H];
  uint32_t wn[H], rk[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    thr[k] = job.thr[k];
    thr_key[k] = group_key(thr[k]);
    wn[k] = 0;
    rk[k] = fl % uint32_t(k + 1);
  }

  const bool live = f0 < n_bins;
  const uint64_t live_lanes = __ballot(live);
  const uint32_t live_bits = live ? (1u << min(n_bins - fl, 8u)) - 1u : 0u;
  const uint32_t r_stop = apart && __ballot(fl + 8u > n_bins) != 0 ? r_last - 1u : r_last;
  if (int(r_begin) <= int(r_stop)) {
    RowLoads<H> a, b;
    hsum_load_row<H>(a, fop, n_bins, c, r_begin, fl);
    for (uint32_t r = r_begin;; r += 2) {
      hsum_load_row<H>(b, fop, n_bins, c, min(r + 1, r_stop), fl);
      hsum_row<H>(st, job, a, r, fl, rk, thr, thr_key, live_lanes, live_bits, wn, wave);
      if (r + 1 > r_stop) break;
      hsum_load_row<H>(a, fop, n_bins, c, min(r + 2, r_stop), fl);
      hsum_row<H>(st, job, b, r + 1, fl, rk, thr, thr_key, live_lanes, live_bits, wn, wave);
      if (r + 2 > r_stop) break;
    }
  }
  flush_rest(st, job, wn);
}

// Up to 4 planes are held to the registers of 6 waves per SIMD and 5 to 8 planes to those of 5, at 8 planes as many
// as the LDS allows; 15 and 16 planes to 128 registers: four waves per SIMD in place of three, 1.49 -> 1.30 ms per 8
// trials of 2^20 bins x 85 rows x 16 planes.  9 to 14 planes take what they need: 105 to 136 registers, four waves up
// to 12 planes and three at 13 and 14.
template <int H>
__global__ __launch_bounds__(kHsumThreads) __attribute__((amdgpu_waves_per_eu(H >= 15 ? 4 : H > 8 ? 1 : H > 4 ? 5 : 6))) void hsum_kernel(
    const HsumJob* __restrict__ jobs, uint32_t n_jobs, uint64_t* stamp) {
  put_stamp(stamp);
  __shared__ HsumStage<H> st;
  hsum_block<H>(st, jobs, n_jobs, blockIdx.x);
}

template <int H>
static void launch_hsum_h(const HsumJob* d_jobs, uint32_t n_jobs, uint32_t n_blocks, hipStream_t stream,
                          uint64_t* stamp) {
  hsum_kernel<H><<<n_blocks, kHsumThreads, 0, stream>>>(d_jobs, n_jobs, stamp);
}

hipError_t launch_hsum(const HsumJob* d_jobs, uint32_t n_jobs, uint32_t n_blocks, uint32_t n_harmonics,
                       hipStream_t stream, uint64_t* stamp) {
  if (n_blocks == 0) return hipSuccess;
  switch (n_harmonics) {
    case 1: launch_hsum_h<1>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 2: launch_hsum_h<2>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 3: launch_hsum_h<3>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 4: launch_hsum_h<4>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 5: launch_hsum_h<5>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 6: launch_hsum_h<6>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 7: launch_hsum_h<7>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 8: launch_hsum_h<8>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 9: launch_hsum_h<9>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 10: launch_hsum_h<10>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 11: launch_hsum_h<11>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 12: launch_hsum_h<12>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 13: launch_hsum_h<13>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 14: launch_hsum_h<14>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 15: launch_hsum_h<15>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    case 16: launch_hsum_h<16>(d_jobs, n_jobs, n_blocks, stream, stamp); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Fused launch: FT convolution of one group with 1024-point tiles and the
// harmonic summing of the group before it
// ---------------------------------------------------------------------------

// Workgroup v is either an FT-convolution work item or a summing block; the
// two kinds are interleaved evenly over the grid (v is an FT item iff
// floor((v+1) A / (A+B)) > floor(v A / (A+B)) for A items and B blocks), so
// the hardware's in-order dispatch keeps both in flight together: the
// VALU-bound transforms and the HBM-bound summing share every CU instead of
// taking turns.  The summing reads a FOP that an earlier launch wrote, so no
// workgroup waits on another.  LDS is one buffer viewed as either kind's.
template <int H>
union FusedLds {
  Ftc1kLds ftc;
  HsumStage<H> hsum;
};

template <int H>
__global__ __launch_bounds__(64 * kFtc1kWaves) __attribute__((amdgpu_waves_per_eu(3, 3))) void fused1k_kernel(
    const FtcJob* __restrict__ ftc_jobs, uint32_t n_ftc_jobs, uint32_t n_items, const float2* __restrict__ tw1,
    const float2* __restrict__ tw2, const HsumJob* __restrict__ hsum_jobs, uint32_t n_hsum_jobs,
    uint32_t n_blocks) {
  static_assert(kHsumThreads == 64 * kFtc1kWaves, "both kinds of work use the same workgroup size");
  __shared__ FusedLds<H> lds;
  const uint32_t v = blockIdx.x;
  const uint64_t total = uint64_t(n_items) + n_blocks;
  const uint32_t a0 = uint32_t(uint64_t(v) * n_items / total);
  const uint32_t a1 = uint32_t(uint64_t(v + 1) * n_items / total);
  if (a1 > a0) {
    WaveFFT1k<true> fft;
    fft.load_twiddles(tw1, tw2, lds.ftc.w2s, int(threadIdx.x) & 63, (threadIdx.x >> 6) == 0);
    ftc1k_item(lds.ftc, fft, ftc_jobs, n_ftc_jobs, a0);
  } else {
    hsum_block<H>(lds.hsum, hsum_jobs, n_hsum_jobs, v - a0);
  }
}

// 16 planes stay unfused when a row length is not a multiple of 8: the fused kernel's transform
// rounds differently from ftconv1w_kernel's, so a plan's choice between them is part of its results.
bool fused_supported(uint32_t tile, uint32_t n_harmonics, bool whole_groups) {
  return tile == 1024 && (n_harmonics == 8 || (n_harmonics == 16 && whole_groups));
}

hipError_t launch_fused(const FtcJob* ftc_jobs, uint32_t n_ftc_jobs, uint32_t n_items, const float2* tw1,
                        const float2* tw2, const HsumJob* hsum_jobs, uint32_t n_hsum_jobs, uint32_t n_blocks,
                        uint32_t n_harmonics, hipStream_t stream) {
  const uint32_t grid = n_items + n_blocks;
  if (grid == 0) return hipSuccess;
  const dim3 block(64 * kFtc1kWaves);
#define FDAS_FUSED(HH)                                                                                         \
  hipLaunchKernelGGL(fused1k_kernel<HH>, dim3(grid), block, 0, stream, ftc_jobs, n_ftc_jobs, n_items, tw1, tw2, \
                     hsum_jobs, n_hsum_jobs, n_blocks)
  if (n_harmonics == 8) FDAS_FUSED(8);
  else if (n_harmonics == 16) FDAS_FUSED(16);
  else return hipErrorInvalidValue;
#undef FDAS_FUSED
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void hplane_kernel(const float* __restrict__ fop, uint32_t n_bins,
                                                     uint32_t n_templates, uint32_t row_begin, uint32_t k_max,
                                                     float* __restrict__ out) {
  const uint32_t f = blockIdx.x * 256u + threadIdx.x;
  const uint32_t r = row_begin + blockIdx.y;
  if (f >= n_bins) return;
  const int c = int(n_templates / 2);
  const int t = int(r) - c;
  float hp = fop[size_t(r) * n_bins + f];
  for (uint32_t k = 2; k <= k_max; ++k) {
    const int rk = c + t / int(k);
    hp += fop[size_t(rk) * n_bins + f / k];
  }
  out[size_t(r) * n_bins + f] = hp;
}

hipError_t launch_hplane(const float* fop, uint32_t n_bins, uint32_t n_templates, uint32_t row_begin, uint32_t n_rows,
                         uint32_t k, float* out, hipStream_t stream) {
  if (n_rows == 0 || n_bins == 0) return hipSuccess;
  dim3 grid((n_bins + 255) / 256, n_rows);
  hipLaunchKernelGGL(hplane_kernel, grid, dim3(256), 0, stream, fop, n_bins, n_templates, row_begin, k, out);
  return hipGetLastError();
}

// Largest HP_k, k = 1..H, of each block of 256 bins x kHmaxRows rows of rows
// [row_begin, row_begin + n_rows): out[k-1][block], block = row group * bin
// blocks + bin block.  HP_k is summed in FP32 in k order, as in hsum_kernel, so
// the values are the ones the summing kernel thresholds.
//
// Bound like the summing kernel, whose loads and sums it uses: a workgroup takes
// 2048 bins, a thread 8 of them, with a maximum per plane in registers.  (One
// bin per thread and a run-time number of planes took 215 us per 2^18 bins x 85
// rows x 8 planes; this takes 30.)
constexpr uint32_t kHmaxRows = 8;
constexpr uint32_t kHmaxBins = 256;

template <int H>
__global__ __launch_bounds__(kHsumThreads) void hmax_kernel(const float* __restrict__ fop, uint32_t n_bins,
                                                            uint32_t n_templates, uint32_t row_begin, uint32_t n_rows,
                                                            float* __restrict__ out) {
  constexpr uint32_t kBlocks = uint32_t(kHsumBinsPerBlock) / kHmaxBins;  // per workgroup
  __shared__ uint32_t red[H][kBlocks];                                   // order keys
  const uint32_t tid = threadIdx.x, block_f0 = blockIdx.x * uint32_t(kHsumBinsPerBlock);
  const uint32_t r0 = row_begin + blockIdx.y * kHmaxRows;
  const uint32_t r_last = min(r0 + kHmaxRows, row_begin + n_rows) - 1;
  const int c = int(n_templates / 2);
  for (uint32_t i = tid; i < H * kBlocks; i += kHsumThreads)
    (&red[0][0])[i] = order_key(__float_as_uint(-INFINITY));
  __syncthreads();
  // One bin of one row (the bins that the 16-byte loads cannot cover, as in hsum_block).
  auto one_bin = [&](uint32_t r, uint32_t f) {
    const int t = int(r) - c;
    float hp = gld(fop, size_t(r) * n_bins + f);
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      if (k > 1) hp += gld(fop, size_t(c + t / k) * n_bins + f / uint32_t(k));
      atomicMax(&red[k - 1][(f - block_f0) / kHmaxBins], order_key(__float_as_uint(fmaxf(-INFINITY, hp))));
    }
  };
  if (n_bins < uint32_t(kHsumBinsPerThread)) {
    if (tid < n_bins)
      for (uint32_t r = r0; r <= r_last; ++r) one_bin(r, tid);
  } else {
    constexpr uint32_t kWaveBins = 64u * kHsumBinsPerThread;
    const uint32_t tail_f0 = (n_bins - 1u) / kWaveBins * kWaveBins;
    const bool apart =
        n_bins % 8u != 0 && r_last + 1u == n_templates && tail_f0 - block_f0 < uint32_t(kHsumBinsPerBlock);
    if (apart)
      for (uint32_t f = tail_f0 + tid; f < min(tail_f0 + kWaveBins, n_bins); f += kHsumThreads) one_bin(r_last, f);
    const uint32_t f0 = block_f0 + tid * uint32_t(kHsumBinsPerThread);
    const uint32_t fl = min(f0, (n_bins - 1u) & ~7u);
    const uint32_t live = f0 < n_bins ? min(n_bins - f0, 8u) : 0u;  // bins of this thread in the row
    const uint32_t r_stop = apart && __ballot(fl + 8u > n_bins) != 0 ? r_last - 1u : r_last;
    float mx[H];
    uint32_t rk[H];
#pragma unroll
    for (int k = 0; k < H; ++k) {
      mx[k] = -INFINITY;
      rk[k] = fl % uint32_t(k + 1);
    }
    if (int(r0) <= int(r_stop)) {
      RowLoads<H> a, b;
      auto row_max = [&](const RowLoads<H>& L) {
        float hp[kHsumBinsPerThread];
#pragma unroll
        for (int i = 0; i < kHsumBinsPerThread; ++i) hp[i] = uint32_t(i) < live ? L.m[i] : -INFINITY;
#pragma unroll
        for (int k = 1; k <= H; ++k) {
          if (k > 1) hsum_add_k<H>(k, hp, L, rk);
#pragma unroll
          for (int i = 0; i < kHsumBinsPerThread; ++i) mx[k - 1] = fmaxf(mx[k - 1], hp[i]);
        }
      };
      hsum_load_row<H>(a, fop, n_bins, c, r0, fl);
      for (uint32_t r = r0;; r += 2) {
        hsum_load_row<H>(b, fop, n_bins, c, min(r + 1, r_stop), fl);
        row_max(a);
        if (r + 1 > r_stop) break;
        hsum_load_row<H>(a, fop, n_bins, c, min(r + 2, r_stop), fl);
        row_max(b);
        if (r + 2 > r_stop) break;
      }
    }
#pragma unroll
    for (int k = 0; k < H; ++k) {
      float v = mx[k];
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
      if ((tid & 31u) == 0) atomicMax(&red[k][tid / 32u], order_key(__float_as_uint(v)));
    }
  }
  __syncthreads();
  const uint32_t bx = (n_bins + kHmaxBins - 1) / kHmaxBins, first = blockIdx.x * kBlocks;
  const size_t nb = size_t(bx) * gridDim.y;
  for (uint32_t i = tid; i < H * kBlocks; i += kHsumThreads) {
    const uint32_t k = i / kBlocks, x = first + i % kBlocks;
    if (x < bx) gst(out, k * nb + size_t(blockIdx.y) * bx + x, __uint_as_float(order_key_inv(red[k][i % kBlocks])));
  }
}

uint32_t hmax_blocks(uint32_t n_bins, uint32_t n_rows) {
  return (n_bins + kHmaxBins - 1) / kHmaxBins * ((n_rows + kHmaxRows - 1) / kHmaxRows);
}

template <int H = 1>
static bool launch_hmax_h(uint32_t n_harmonics, dim3 grid, hipStream_t stream, const float* fop, uint32_t n_bins,
                          uint32_t n_templates, uint32_t row_begin, uint32_t n_rows, float* out) {
  if constexpr (H <= int(kMaxHarmonics)) {
    if (n_harmonics != uint32_t(H))
      return launch_hmax_h<H + 1>(n_harmonics, grid, stream, fop, n_bins, n_templates, row_begin, n_rows, out);
    hipLaunchKernelGGL(hmax_kernel<H>, grid, dim3(kHsumThreads), 0, stream, fop, n_bins, n_templates, row_begin,
                       n_rows, out);
    return true;
  }
  return false;
}

hipError_t launch_hmax(const float* fop, uint32_t n_bins, uint32_t n_templates, uint32_t row_begin, uint32_t n_rows,
                       uint32_t n_harmonics, float* out, hipStream_t stream) {
  if (n_rows == 0 || n_bins == 0) return hipSuccess;
  dim3 grid((n_bins + kHsumBinsPerBlock - 1) / kHsumBinsPerBlock, (n_rows + kHmaxRows - 1) / kHmaxRows);
  if (!launch_hmax_h(n_harmonics, grid, stream, fop, n_bins, n_templates, row_begin, n_rows, out))
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Selection: keep the `cap` strongest detections of a plane (ties: smaller
// (row, bin) key first), returned sorted by key.
// ---------------------------------------------------------------------------

// Inclusive prefix sum over the wave: row shifts inside each row of 16 lanes,
// then the rows' totals broadcast upwards (VALU only; six LDS permutes take
// about ten times as long).
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x111, 0xf, 0xf, false));  // row_shr:1
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x112, 0xf, 0xf, false));  // row_shr:2
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x114, 0xf, 0xf, false));  // row_shr:4
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x118, 0xf, 0xf, false));  // row_shr:8
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1, 3
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2, 3
  return v;
}

// Exclusive prefix sum over a workgroup of THREADS threads.  s_waves: one LDS
// word per wave, not reused before the caller's next barrier.
template <int THREADS>
__device__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_waves) {
  constexpr uint32_t n_waves = THREADS / 64;
  static_assert(n_waves <= 16, "the waves' totals are scanned in one row of lanes");
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  const uint32_t x = wave_inclusive_scan(v);
  if (lane == 63) s_waves[wave] = x;
  __syncthreads();
  const uint32_t w = lane < n_waves ? s_waves[lane] : 0u;
  const uint32_t before = wave_inclusive_scan(w) - w;  // lane i: total of waves 0 .. i-1
  return x - v + uint32_t(__builtin_amdgcn_readlane(int(before), __builtin_amdgcn_readfirstlane(int(wave))));
}

// Cut bin b*: the highest bin whose suffix count sum_{b >= b*} hist[b] reaches
// `cap`.  s_out[0] = b*, s_out[1] = entries strictly above b*.  The histogram
// counts every spilled entry and there are more than `cap` of them, so a cut
// exists; the defaults (bin 0, nothing above) keep b* inside the histogram
// regardless.
template <int THREADS, class Bin>
__device__ void find_cut(Bin hist_bin, uint32_t cap, uint32_t* s_waves, uint32_t* s_out) {
  constexpr int PER = int(kSelectBins) / THREADS;
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_out[0] = 0;
    s_out[1] = 0;
  }
  uint32_t h[PER];
  uint32_t local = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    h[j] = hist_bin(kSelectBins - 1 - uint32_t(tid * PER + j));
    local += h[j];
  }
  const uint32_t excl = block_exclusive_scan<THREADS>(local, s_waves);
  uint32_t bin, above;
  if (cut_in_share<PER>(h, excl, cap, uint32_t(tid * PER), &bin, &above)) {
    s_out[0] = bin;
    s_out[1] = above;
  }
  __syncthreads();
}

// Planes of no more detections than the compact list holds are left to the last kernel, which reads the spill list
// itself; for them the histogram and the compaction are two empty kernels.  With that and sort_by_runs the selection
// of 8 planes of cap 512 takes 11 us at 4,999 bins x 33 templates and 12 at 32,768 x 85; it took 22 and 18.
__device__ __forceinline__ bool select_direct(const SelectJob& job, uint32_t n) { return n <= job.compact_cap; }

__global__ __launch_bounds__(256) void cand_hist_kernel(const SelectJob* __restrict__ jobs, uint64_t* stamp) {
  put_stamp(stamp);
  const SelectJob& job = jobs[blockIdx.y];
  const uint32_t n = min(gld(job.count, 0), job.spill_cap);
  if (select_direct(job, n)) return;
  __shared__ uint32_t h[kSelectBins];
  const int tid = threadIdx.x;
  for (uint32_t i = tid; i < kSelectBins; i += 256) h[i] = 0;
  __syncthreads();
  const uint32_t tb = histogram_base(__float_as_uint(job.thr));
  const uint32_t per = (n + kSelectSlices - 1) / kSelectSlices;
  const uint32_t beg = blockIdx.x * per, end = min(beg + per, n);
  const float* __restrict__ pw = job.spill_pwr;
  for (uint32_t e0 = beg; e0 < end; e0 += 4 * 256) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t e = e0 + uint32_t(u * 256 + tid);
      v[u] = e < end ? __float_as_uint(gld(pw, e)) : 0xffffffffu;  // all ones: past the slice
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (v[u] != 0xffffffffu) atomicAdd(&h[power_bin(v[u], tb)], 1u);
  }
  __syncthreads();
  for (uint32_t i = tid; i < kSelectBins; i += 256)
    if (h[i]) gatomic_add(job.hist + i, h[i]);
}

// Slots for the lanes that set take[u], u = 0 .. U-1, from a counter in LDS, with
// one atomic per wave; slot[u] is meaningful where take[u] is set.
template <int U>
__device__ __forceinline__ void wave_append(uint32_t* counter, const bool (&take)[U], uint32_t (&slot)[U]) {
  uint64_t mask[U];
  uint32_t total = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    mask[u] = __ballot(take[u]);
    slot[u] = total + lanes_below(mask[u]);
    total += uint32_t(__builtin_popcountll(mask[u]));
  }
  if (total == 0) return;
  uint32_t base = 0;
  if (lane_id() == 0) base = atomicAdd(counter, total);
  base = __shfl(base, 0);
#pragma unroll
  for (int u = 0; u < U; ++u) slot[u] += base;
}

// Copies the entries at or above the cut bin to the compact list.  Bound by
// latency: a workgroup collects its slice's entries in LDS and reserves their
// place in the list with one global atomic per flush.  (One returning global
// atomic per wave with a hit, on the plane's one counter, made 2,500 of them
// queue up for plane 1 of a 2^21-bin trial: 43 us per launch of 8 planes,
// against 10 this way.)
__global__ __launch_bounds__(256) void cand_compact_kernel(const SelectJob* __restrict__ jobs) {
  const SelectJob& job = jobs[blockIdx.y];
  const uint32_t n = min(gld(job.count, 0), job.spill_cap);
  if (select_direct(job, n)) return;
  constexpr uint32_t kStep = 4 * 256, kStage = 2 * kStep;
  __shared__ uint32_t waves[4];
  __shared__ uint32_t cut[2];
  __shared__ uint32_t key[kStage];
  __shared__ float pwr[kStage];
  __shared__ uint32_t n_staged, g_base;
  const int tid = threadIdx.x;
  if (tid == 0) n_staged = 0;
  find_cut<256>([&](uint32_t b) { return gld(job.hist, b); }, job.cap, waves, cut);
  const uint32_t bstar = cut[0];
  const uint32_t tb = histogram_base(__float_as_uint(job.thr));
  const uint32_t per = (n + kSelectSlices - 1) / kSelectSlices;
  const uint32_t beg = blockIdx.x * per, end = min(beg + per, n);
  for (uint32_t e0 = beg; e0 < end; e0 += kStep) {
    uint32_t k[4];
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t e = min(e0 + uint32_t(u * 256 + tid), end - 1u);
      v[u] = gld(job.spill_pwr, e);
      k[u] = gld(job.spill_key, e);
    }
    bool sel[4];
    uint32_t pos[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      sel[u] = e0 + uint32_t(u * 256 + tid) < end && power_bin(__float_as_uint(v[u]), tb) >= bstar;
    wave_append(&n_staged, sel, pos);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (!sel[u]) continue;
      key[pos[u]] = k[u];
      pwr[pos[u]] = v[u];
    }
    __syncthreads();
    const uint32_t staged = n_staged;
    __syncthreads();  // everyone has read it
    if (staged > kStage - kStep || e0 + kStep >= end) {  // no room for another step, or done
      if (tid == 0) {
        g_base = staged ? gatomic_add(job.compact_n, staged) : 0u;
        n_staged = 0;
      }
      __syncthreads();
      const uint32_t base = g_base;
      for (uint32_t i = tid; i < staged && base + i < job.compact_cap; i += 256) {
        gst(job.compact_key, base + i, key[i]);
        gst(job.compact_pwr, base + i, pwr[i]);
      }
    }
    __syncthreads();
  }
}

constexpr int kSortBins = 256;  // values of one sort digit

// LDS of one selection workgroup: up to CAP kept entries; the pool of the cut
// bin's entries, the radix-select histogram and the sort's digit counters are
// never live together.
template <int THREADS, int CAP>
struct SelectShared {
  static constexpr int kWaves = THREADS / 64;
  static constexpr int kRow = kSortBins + 1;  // row stride of the counters: spreads a digit's over the banks
  uint32_t key[CAP];
  float pwr[CAP];
  union {
    uint64_t pool[kSelectPool];
    uint32_t hist[2048];
    uint32_t digit[kWaves * kRow];
  };
  uint32_t waves[kWaves];
  uint32_t misc[8];
};

// One radix-select digit pass: among values v with (v & mask) == prefix, find
// the digit (bits [shift, shift+width)) holding the `rank`-th element counted
// from the top (descending) or bottom (ascending).  Updates prefix/mask/rank.
template <bool DESCENDING, int THREADS, class Shared, typename Get>
__device__ void radix_pass(Shared& sh, uint32_t n, Get get, uint32_t shift, uint32_t width, uint32_t& prefix,
                           uint32_t& mask, uint32_t& rank) {
  constexpr int PER = 2048 / THREADS;
  const int tid = threadIdx.x;
  const uint32_t nb = 1u << width;
  for (uint32_t i = tid; i < 2048; i += THREADS) sh.hist[i] = 0;
  __syncthreads();
  for (uint32_t e0 = tid; e0 < n; e0 += 4 * THREADS) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = get(min(e0 + uint32_t(u * THREADS), n - 1u));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (e0 + uint32_t(u * THREADS) < n && (v[u] & mask) == prefix) atomicAdd(&sh.hist[(v[u] >> shift) & (nb - 1)], 1u);
  }
  __syncthreads();
  // Thread t owns ordered positions u = PER t .. PER t + PER - 1 (u counts from the selected end).
  uint32_t h[PER], local = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t u = uint32_t(PER * tid + j);
    const uint32_t d = DESCENDING ? (nb - 1 - u) : u;
    h[j] = u < nb ? sh.hist[d] : 0u;
    local += h[j];
  }
  const uint32_t excl = block_exclusive_scan<THREADS>(local, sh.waves);
  uint32_t acc = excl;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (acc < rank && rank <= acc + h[j]) {
      const uint32_t u = uint32_t(PER * tid + j);
      sh.misc[0] = DESCENDING ? (nb - 1 - u) : u;
      sh.misc[1] = rank - acc;
      sh.misc[2] = h[j];
    }
    acc += h[j];
  }
  __syncthreads();
  prefix |= sh.misc[0] << shift;
  mask |= (nb - 1) << shift;
  rank = sh.misc[1];
  __syncthreads();
}

// v of the lane whose index differs in the bits of M.
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  if constexpr (M == 1) return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0xb1, 0xf, 0xf, true));  // quad_perm
  if constexpr (M == 2) return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x4e, 0xf, 0xf, true));
  if constexpr (M == 8) return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x128, 0xf, 0xf, true));  // row_ror:8
  if constexpr (M == 4 || M == 16) return uint32_t(__builtin_amdgcn_ds_swizzle(int(v), (M << 10) | 0x1f));
  return uint32_t(__shfl_xor(int(v), M));
}

// Bitonic sort of a wave's 64 K keys, ascending; lane l holds entries K l .. K l + K - 1.
template <int K, int SIZE = 2, int STRIDE = 1>
__device__ __forceinline__ void wave_sort(uint32_t (&a)[K]) {
  if constexpr (SIZE <= 64 * K) {
    const uint32_t lane = lane_id();
    if constexpr (STRIDE >= K) {
      constexpr int M = STRIDE / K;
      const bool keep_min = ((lane & M) == 0) == ((lane & (SIZE / K)) == 0);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const uint32_t other = lane_xor<M>(a[k]);
        a[k] = keep_min ? min(a[k], other) : max(a[k], other);
      }
    } else {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (k & STRIDE) continue;
        const bool up = SIZE < K ? (k & SIZE) == 0 : (lane & (SIZE / K)) == 0;
        const uint32_t lo = min(a[k], a[k + STRIDE]), hi = max(a[k], a[k + STRIDE]);
        a[k] = up ? lo : hi;
        a[k + STRIDE] = up ? hi : lo;
      }
    }
    if constexpr (STRIDE > 1) wave_sort<K, SIZE, STRIDE / 2>(a);
    else wave_sort<K, SIZE * 2, SIZE>(a);
  }
}

// Sorts n <= 64 K entries per wave by key (all different), ascending.  Each wave sorts its entries' keys in
// registers, and an entry's place is the number of smaller keys in every wave's run, by binary searches: 3 barriers,
// where the radix sort takes 7 a pass.  For workgroups of 4 waves: 512 entries in about 2 us against 5 (3 passes) and
// 6.7 (4 passes); the searches grow with the number of runs, and 16 runs of 256 would take longer than the passes.
template <int K, int THREADS, class Shared>
__device__ void sort_by_runs(Shared& sh, uint32_t n) {
  constexpr uint32_t RUN = 64 * K;
  uint32_t* runs = reinterpret_cast<uint32_t*>(sh.pool);
  uint32_t key[K], sorted[K], place[K];
  float pwr[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t i = threadIdx.x * K + uint32_t(k);
    key[k] = i < n ? sh.key[i] : 0xffffffffu;
    pwr[k] = i < n ? sh.pwr[i] : 0.f;
    sorted[k] = key[k];
    place[k] = 0;
  }
  wave_sort<K>(sorted);
#pragma unroll
  for (int k = 0; k < K; ++k) runs[threadIdx.x * K + uint32_t(k)] = sorted[k];
  __syncthreads();
#pragma unroll
  for (uint32_t w = 0; w < THREADS / 64; ++w) {
    const uint32_t* run = runs + w * RUN;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      uint32_t c = 0;  // keys of the run below this one
#pragma unroll
      for (uint32_t s = RUN / 2; s > 0; s /= 2) c += run[c + s - 1] < key[k] ? s : 0u;
      place[k] += c + (run[c] < key[k] ? 1u : 0u);
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (threadIdx.x * K + uint32_t(k) >= n) continue;
    sh.key[place[k]] = key[k];
    sh.pwr[place[k]] = pwr[k];
  }
}

// Sorts the n kept entries by key (row, bin), ascending: a radix sort in place,
// 8 bits a pass, over the bits that rows and bins really use (3 passes for a
// spectrum of 2^17 bins and 85 templates, 4 for 2^21).  Bound by LDS latency and
// barriers: an entry's place is its digit's start, plus what earlier waves and
// the wave's earlier entries hold of that digit (one match by ballots), so a
// pass takes 7 barriers, where the bitonic network took one for each of its 78
// steps over 4096 entries.
template <int THREADS, int CAP, class Shared>
__device__ void sort_by_key(Shared& sh, uint32_t n) {
  constexpr int E = CAP / THREADS, NW = THREADS / 64, ROW = Shared::kRow;
  constexpr int PER = kSortBins * NW / THREADS;  // counters one thread scans
  static_assert(PER * THREADS == kSortBins * NW, "whole counters per thread");
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const uint32_t sub = (n + THREADS - 1) / THREADS;  // 64-entry runs of one wave
  uint32_t key[E], place[E];
  float pwr[E];
  // Bits in use: bins below 2^nb, rows above them.
  if (tid < 2) sh.misc[4 + tid] = 0;
  __syncthreads();
  uint32_t or_bin = 0, or_row = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const uint32_t i = (wave * sub + uint32_t(e)) * 64 + lane;
    key[e] = 0;
    pwr[e] = 0.f;
    place[e] = 0;
    if (uint32_t(e) < sub && i < n) {
      key[e] = sh.key[i];
      pwr[e] = sh.pwr[i];
      or_bin |= key[e] & ((1u << kKeyBinBits) - 1u);
      or_row |= key[e] >> kKeyBinBits;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    or_bin |= __shfl_xor(or_bin, o);
    or_row |= __shfl_xor(or_row, o);
  }
  if (lane == 0) {
    atomicOr(&sh.misc[4], or_bin);
    atomicOr(&sh.misc[5], or_row);
  }
  __syncthreads();
  const uint32_t nb = 32u - uint32_t(__builtin_clz(sh.misc[4] | 1u));
  const uint32_t bits = nb + 32u - uint32_t(__builtin_clz(sh.misc[5] | 1u));
  const uint32_t passes = (bits + 7u) / 8u, width = (bits + passes - 1u) / passes;  // digits of equal width, <= 8 bits
  auto digit_of = [&](uint32_t k, uint32_t shift) {
    const uint32_t packed = ((k >> kKeyBinBits) << nb) | (k & ((1u << kKeyBinBits) - 1u));
    return (packed >> shift) & ((1u << width) - 1u);
  };
  uint32_t* mine = sh.digit + wave * ROW;
  for (uint32_t shift = 0; shift < bits; shift += width) {
    for (uint32_t i = tid; i < uint32_t(NW * ROW); i += THREADS) sh.digit[i] = 0;
    __syncthreads();
    // Lanes of the run that hold the same digit (its bits' ballots, complemented where the lane's bit is 0).
    uint32_t same_lo[E], same_hi[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint64_t valid = __ballot(uint32_t(e) < sub && (wave * sub + uint32_t(e)) * 64 + lane < n);
      same_lo[e] = uint32_t(valid);
      same_hi[e] = uint32_t(valid >> 32);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (uint32_t(j) >= width) break;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int bit = -int((digit_of(key[e], shift) >> j) & 1u);  // all ones or zero
        const uint64_t m = __ballot(bit != 0);
        same_lo[e] &= ~(uint32_t(m) ^ uint32_t(bit));
        same_hi[e] &= ~(uint32_t(m >> 32) ^ uint32_t(bit));
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (uint32_t(e) >= sub) break;
      const bool valid = (wave * sub + uint32_t(e)) * 64 + lane < n;
      const uint32_t d = digit_of(key[e], shift);
      const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi[e], __builtin_amdgcn_mbcnt_lo(same_lo[e], 0u));
      const uint32_t before = mine[d];
      wave_lds_order();
      place[e] = before + below;
      if (valid && below == 0)
        mine[d] = before + uint32_t(__builtin_popcount(same_lo[e])) + uint32_t(__builtin_popcount(same_hi[e]));
      wave_lds_order();
    }
    __syncthreads();
    uint32_t c[PER], local = 0;  // digit-major: all waves' counters of digit 0, of digit 1, ...
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t q = tid * PER + uint32_t(j);
      c[j] = sh.digit[(q % NW) * ROW + q / NW];
      local += c[j];
    }
    uint32_t acc = block_exclusive_scan<THREADS>(local, sh.waves);
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t q = tid * PER + uint32_t(j);
      sh.digit[(q % NW) * ROW + q / NW] = acc;
      acc += c[j];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (uint32_t(e) >= sub || (wave * sub + uint32_t(e)) * 64 + lane >= n) continue;
      const uint32_t pos = mine[digit_of(key[e], shift)] + place[e];
      sh.key[pos] = key[e];
      sh.pwr[pos] = pwr[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint32_t i = (wave * sub + uint32_t(e)) * 64 + lane;
      if (uint32_t(e) >= sub || i >= n) continue;
      key[e] = sh.key[i];
      pwr[e] = sh.pwr[i];
    }
  }
}

template <int THREADS>
__device__ void bitonic_sort_u64(uint64_t* a, uint32_t n) {
  const int tid = threadIdx.x;
  uint32_t p2 = 1;
  while (p2 < n) p2 <<= 1;
  for (uint32_t i = n + tid; i < p2; i += THREADS) a[i] = ~0ull;
  __syncthreads();
  for (uint32_t k = 2; k <= p2; k <<= 1) {
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      for (uint32_t i = tid; i < p2; i += THREADS) {
        const uint32_t ixj = i ^ j;
        if (ixj > i) {
          const uint64_t x = a[i], y = a[ixj];
          if ((x > y) == ((i & k) == 0)) {
            a[i] = y;
            a[ixj] = x;
          }
        }
      }
      __syncthreads();
    }
  }
}

// Appends the `take` smallest of the pool's n entries (power descending, then
// key ascending) to the kept list from `at` on.  A few hundred entries, the
// usual size of the cut bin, are ranked by counting; a pool beyond
// kCountedPool, where that would cost more than it saves (n^2 / THREADS
// compares), is sorted.
constexpr uint32_t kCountedPool = 1024;

template <int THREADS, class Shared>
__device__ void take_from_pool(Shared& sh, uint32_t n, uint32_t take, uint32_t at) {
  const uint32_t tid = threadIdx.x;
  auto keep = [&](uint32_t slot, uint64_t v) {
    sh.key[slot] = uint32_t(v);
    sh.pwr[slot] = __uint_as_float(order_key_inv(~uint32_t(v >> 32)));
  };
  if (n > kCountedPool) {
    bitonic_sort_u64<THREADS>(sh.pool, n);
    for (uint32_t i = tid; i < take && i < n; i += THREADS) keep(at + i, sh.pool[i]);
    return;
  }
  for (uint32_t i = tid; i < n; i += THREADS) {
    const uint64_t v = sh.pool[i];
    uint32_t rank = 0;
#pragma unroll 8
    for (uint32_t q = 0; q < n; ++q) rank += sh.pool[q] < v ? 1u : 0u;
    if (rank < take) keep(at + rank, v);
  }
}

// Exact top-`cap` of the whole spill by radix select on (power desc, key asc).
// Used when the boundary bin holds more entries than the LDS pool.
template <int THREADS, class Shared>
__device__ uint32_t radix_select_spill(Shared& sh, const SelectJob& job, uint32_t n) {
  const int tid = threadIdx.x;
  const uint32_t cap = job.cap;
  const uint32_t* __restrict__ skey = job.spill_key;
  const float* __restrict__ spwr = job.spill_pwr;
  auto pkey = [&](uint32_t e) { return order_key(__float_as_uint(gld(spwr, e))); };
  uint32_t prefix = 0, mask = 0, rank = cap;
  radix_pass<true, THREADS>(sh, n, pkey, 21, 11, prefix, mask, rank);
  radix_pass<true, THREADS>(sh, n, pkey, 10, 11, prefix, mask, rank);
  radix_pass<true, THREADS>(sh, n, pkey, 0, 10, prefix, mask, rank);
  const uint32_t vkey = prefix;  // order key of the cap-th strongest power V
  const uint32_t n_equal = sh.misc[2];
  // `rank` entries with power == V are kept: the smallest keys among them.
  uint32_t kmax = 0xffffffffu;
  if (n_equal > rank) {
    auto kbits = [&](uint32_t e) { return pkey(e) == vkey ? gld(skey, e) : 0xffffffffu; };
    uint32_t kp = 0, km = 0, kr = rank;
    radix_pass<false, THREADS>(sh, n, kbits, 21, 11, kp, km, kr);
    radix_pass<false, THREADS>(sh, n, kbits, 10, 11, kp, km, kr);
    radix_pass<false, THREADS>(sh, n, kbits, 0, 10, kp, km, kr);
    kmax = kp;
  }
  if (tid == 0) sh.misc[3] = 0;
  __syncthreads();
  for (uint32_t e = tid; e < n; e += THREADS) {
    const float pv = gld(spwr, e);
    const uint32_t pk = order_key(__float_as_uint(pv));
    const uint32_t key = gld(skey, e);
    if (pk > vkey || (pk == vkey && key <= kmax)) {
      const uint32_t pos = atomicAdd(&sh.misc[3], 1u);
      if (pos < cap) {
        sh.key[pos] = key;
        sh.pwr[pos] = pv;
      }
    }
  }
  __syncthreads();
  return min(sh.misc[3], cap);
}

// One workgroup per plane: the kept entries, sorted.  CAP >= the job's cap.
// Bound by latency (one workgroup's barriers and LDS round trips): 19 us for 8
// planes that keep 4096 of 70,000 .. 173,000 entries, 13.6 of them in the sort (with
// bitonic sorts of key and power 75).  Results in host memory need no fence of the
// kernel's own: the stream's or event's synchronisation makes them visible, and the
// fence, which writes back the L2, took 2 to 4 us.
template <int THREADS, int CAP>
__global__ __launch_bounds__(THREADS) void select_final_kernel(const SelectJob* __restrict__ jobs, uint64_t* ends) {
  __shared__ SelectShared<THREADS, CAP> sh;
  const SelectJob& job = jobs[blockIdx.x];
  const int tid = threadIdx.x;
  const uint32_t detected = gld(job.count, 0), n = min(detected, job.spill_cap);
  const uint32_t cap = job.cap;

  uint32_t kept;
  if (n <= cap) {
    for (uint32_t e = tid; e < n; e += THREADS) {
      sh.key[e] = gld(job.spill_key, e);
      sh.pwr[e] = gld(job.spill_pwr, e);
    }
    kept = n;
  } else {
    constexpr int U = THREADS == 256 ? 8 : 4;  // loads in flight per thread
    const uint32_t tb = histogram_base(__float_as_uint(job.thr));
    const bool direct = select_direct(job, n);
    if (direct) {
      for (uint32_t i = tid; i < kSelectBins; i += THREADS) sh.hist[i] = 0;
      __syncthreads();
      for (uint32_t e0 = tid; e0 < n; e0 += U * THREADS) {
        uint32_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __float_as_uint(gld(job.spill_pwr, min(e0 + uint32_t(u * THREADS), n - 1u)));
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (e0 + uint32_t(u * THREADS) < n) atomicAdd(&sh.hist[power_bin(v[u], tb)], 1u);
      }
      __syncthreads();
      find_cut<THREADS>([&](uint32_t b) { return sh.hist[b]; }, cap, sh.waves, sh.misc);
    } else {
      find_cut<THREADS>([&](uint32_t b) { return gld(job.hist, b); }, cap, sh.waves, sh.misc);
    }
    const uint32_t bstar = sh.misc[0], above = sh.misc[1];
    const uint32_t m = direct ? n : gld(job.compact_n, 0);
    const uint32_t pool_n = direct ? sh.hist[bstar] : gld(job.hist, bstar);
    const uint32_t* list_key = direct ? job.spill_key : job.compact_key;
    const float* list_pwr = direct ? job.spill_pwr : job.compact_pwr;
    __syncthreads();
    if (m <= job.compact_cap && pool_n <= kSelectPool && above < cap) {
      if (tid == 0) {
        sh.misc[3] = 0;
        sh.misc[4] = 0;
      }
      __syncthreads();
      for (uint32_t e0 = 0; e0 < m; e0 += U * THREADS) {
        float v[U];
        uint32_t key[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t e = min(e0 + uint32_t(u * THREADS + tid), m - 1u);
          v[u] = gld(list_pwr, e);
          key[u] = gld(list_key, e);
        }
        bool strong[U], at_cut[U];
        uint32_t pos[U], q[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool in = e0 + uint32_t(u * THREADS + tid) < m;
          const uint32_t bin = power_bin(__float_as_uint(v[u]), tb);
          strong[u] = in && bin > bstar;
          at_cut[u] = in && bin == bstar;
        }
        wave_append(&sh.misc[3], strong, pos);
        wave_append(&sh.misc[4], at_cut, q);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (strong[u] && pos[u] < cap) {
            sh.key[pos[u]] = key[u];
            sh.pwr[pos[u]] = v[u];
          }
          if (at_cut[u] && q[u] < kSelectPool)
            sh.pool[q[u]] = (uint64_t(~order_key(__float_as_uint(v[u]))) << 32) | key[u];  // strongest first
        }
      }
      __syncthreads();
      take_from_pool<THREADS>(sh, min(sh.misc[4], kSelectPool), cap - above, above);
      kept = cap;
    } else {
      kept = radix_select_spill<THREADS>(sh, job, n);
    }
  }
  __syncthreads();
  if constexpr (CAP <= 4 * THREADS && THREADS == 256) {
    if (kept <= THREADS) sort_by_runs<1, THREADS>(sh, kept);
    else if (kept <= 2 * THREADS) sort_by_runs<2, THREADS>(sh, kept);
    else sort_by_runs<4, THREADS>(sh, kept);
  } else {
    sort_by_key<THREADS, CAP>(sh, kept);
  }
  __syncthreads();
  for (uint32_t e = tid; e < kept; e += THREADS) {
    gst(job.out_key, e, sh.key[e]);
    gst(job.out_pwr, e, sh.pwr[e]);
  }
  if (tid == 0) {
    gst(job.out_n, 0, kept);
    gst(job.out_count, 0, detected);
  }
  if (ends && tid == 0) ends[blockIdx.x] = wall_clock64();
}

// ---------------------------------------------------------------------------
// Quantile thresholds: order statistics of a plane
// ---------------------------------------------------------------------------

constexpr int kRankThreads = 1024;
struct RankShared {
  uint32_t hist[2048];
  uint32_t waves[kRankThreads / 64];
  uint32_t misc[8];
};

// The rank-th largest (1 = largest) of the order keys get(0) .. get(n-1), 1 <= rank <= n:
// a radix select from the highest bit in which the keys differ, 11 bits a pass
// (from the sign on, most keys would share their first digit, and its counter).
template <typename Get>
__device__ uint32_t radix_rank(RankShared& sh, uint32_t n, Get get, uint32_t rank) {
  const uint32_t tid = threadIdx.x;
  __syncthreads();  // earlier readers of sh are done
  if (tid == 0) {
    sh.misc[4] = 0;
    sh.misc[5] = 0xffffffffu;
  }
  __syncthreads();
  uint32_t any = 0, all = 0xffffffffu;
  for (uint32_t e0 = tid; e0 < n; e0 += 4 * kRankThreads) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t v = get(min(e0 + uint32_t(u * kRankThreads), n - 1u));
      any |= v;
      all &= v;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    any |= __shfl_xor(any, o);
    all &= __shfl_xor(all, o);
  }
  if (lane_id() == 0) {
    atomicOr(&sh.misc[4], any);
    atomicAnd(&sh.misc[5], all);
  }
  __syncthreads();
  const uint32_t same = sh.misc[5], differ = sh.misc[4] ^ same;
  __syncthreads();
  if (differ == 0) return same;
  uint32_t bits = 32u - uint32_t(__builtin_clz(differ));  // low bits still open
  uint32_t mask = bits < 32u ? ~0u << bits : 0u, prefix = same & mask;
  while (bits > 0) {
    const uint32_t width = min(bits, 11u);
    bits -= width;
    radix_pass<true, kRankThreads>(sh, n, get, bits, width, prefix, mask, rank);
  }
  return prefix;
}

// thr_k just below the want-th largest of plane k's nb block maxima, or -inf when
// there are fewer blocks or that value is not positive: at least `want` values
// of the plane lie above it.  Written into the jobs of the summing pass that follows.
__global__ __launch_bounds__(kRankThreads) void quantile_bound_kernel(const float* __restrict__ maxima, uint32_t nb,
                                                                      uint32_t want, HsumJob* hsum, SelectJob* sel,
                                                                      float* thr_out) {
  __shared__ RankShared sh;
  const uint32_t k = blockIdx.x;
  float thr = -INFINITY;
  if (nb >= want) {
    auto key = [&](uint32_t e) { return order_key(__float_as_uint(gld(maxima, size_t(k) * nb + e))); };
    const uint32_t v = order_key_inv(radix_rank(sh, nb, key, want));
    if (v != 0 && (v & 0x80000000u) == 0) thr = __uint_as_float(v - 1u);
  }
  if (threadIdx.x == 0) {
    hsum->thr[k] = thr;
    sel[k].thr = thr;
    thr_out[k] = thr;
  }
}

// out = counts[H], then the values at the 0-based descending ranks r_lo and r_hi of
// each plane's spilled powers (0 where the spill list does not hold the rank, or overflowed).
__global__ __launch_bounds__(kRankThreads) void quantile_rank_kernel(const SelectJob* __restrict__ jobs, uint32_t r_lo,
                                                                     uint32_t r_hi, uint32_t* __restrict__ out) {
  __shared__ RankShared sh;
  const uint32_t k = blockIdx.x, H = gridDim.x;
  const SelectJob& job = jobs[k];
  const uint32_t n = gld(job.count, 0);
  uint32_t lo = 0, hi = 0;
  if (n <= job.spill_cap && r_lo < n && r_hi < n) {
    auto key = [&](uint32_t e) { return order_key(__float_as_uint(gld(job.spill_pwr, e))); };
    lo = order_key_inv(radix_rank(sh, n, key, r_lo + 1));
    hi = r_hi == r_lo ? lo : order_key_inv(radix_rank(sh, n, key, r_hi + 1));
  }
  if (threadIdx.x == 0) {
    gst(out, k, n);
    gst(out, H + k, lo);
    gst(out, 2 * H + k, hi);
  }
}

hipError_t launch_quantile_bound(const float* maxima, uint32_t nb, uint32_t want, uint32_t n_harmonics, HsumJob* d_hsum,
                                 SelectJob* d_sel, float* thr_out, hipStream_t stream) {
  hipLaunchKernelGGL(quantile_bound_kernel, dim3(n_harmonics), dim3(kRankThreads), 0, stream, maxima, nb, want, d_hsum,
                     d_sel, thr_out);
  return hipGetLastError();
}

hipError_t launch_quantile_rank(const SelectJob* d_sel, uint32_t n_harmonics, uint32_t r_lo, uint32_t r_hi,
                                uint32_t* out, hipStream_t stream) {
  hipLaunchKernelGGL(quantile_rank_kernel, dim3(n_harmonics), dim3(kRankThreads), 0, stream, d_sel, r_lo, r_hi, out);
  return hipGetLastError();
}

hipError_t launch_select(const SelectJob* d_jobs, uint32_t n_jobs, uint32_t cap, hipStream_t stream, uint64_t* stamp,
                         uint64_t* ends) {
  if (n_jobs == 0) return hipSuccess;
  if (cap > kSelectMaxCap) return hipErrorInvalidValue;
  hipLaunchKernelGGL(cand_hist_kernel, dim3(kSelectSlices, n_jobs), dim3(256), 0, stream, d_jobs, stamp);
  hipLaunchKernelGGL(cand_compact_kernel, dim3(kSelectSlices, n_jobs), dim3(256), 0, stream, d_jobs);
  // The workgroup grows with the list.  With 256 / 512 / 1024 threads this kernel takes, for 8 planes and a cap of 512,
  // 9.4 / 11.6 / 10.5 us at 32,768 bins x 85 rows and 8.5 / 12.0 / 11.2 at 2^21; a cap of 1024 12.2 / 12.5 / 10.9 and
  // 11.3 / 13.2 / 12.2, where the small workgroup needs a quarter of the CU beside other kernels; a cap of 2048 at
  // 32,768 bins 25 / 17 / 15; a cap of 4096 at 2^21 42 / 25 / 23.
  if (cap <= 1024) select_final_kernel<256, 1024><<<n_jobs, 256, 0, stream>>>(d_jobs, ends);
  else if (cap <= 4096) select_final_kernel<1024, 4096><<<n_jobs, 1024, 0, stream>>>(d_jobs, ends);
  else select_final_kernel<1024, 8192><<<n_jobs, 1024, 0, stream>>>(d_jobs, ends);
  return hipGetLastError();
}

// The counters and histograms of a group's selection jobs to zero.
__global__ __launch_bounds__(256) void clear_counters_kernel(const SelectJob* __restrict__ jobs) {
  const SelectJob& job = jobs[blockIdx.x];
  for (uint32_t i = threadIdx.x; i < kSelectBins; i += 256) gst(job.hist, i, 0u);
  if (threadIdx.x == 0) {
    gst(job.compact_n, 0, 0u);
    gst(const_cast<uint32_t*>(job.count), 0, 0u);
  }
}

hipError_t launch_clear_counters(const SelectJob* d_jobs, uint32_t n_jobs, hipStream_t stream) {
  if (n_jobs == 0) return hipSuccess;
  hipLaunchKernelGGL(clear_counters_kernel, dim3(n_jobs), dim3(256), 0, stream, d_jobs);
  return hipGetLastError();
}

__global__ void zero_u32_kernel(uint32_t* __restrict__ p, uint32_t n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

hipError_t launch_zero_u32(uint32_t* p, uint32_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const uint32_t blocks = min((n + 255u) / 256u, 1024u);
  hipLaunchKernelGGL(zero_u32_kernel, dim3(blocks), dim3(256), 0, stream, p, n);
  return hipGetLastError();
}

static_assert(sizeof(JobPack) <= 3584, "job descriptors must fit a kernel argument block");

__global__ __launch_bounds__(256) void put_jobs_kernel(JobPack pack, FtcJob* ftc, HsumJob* hsum, SelectJob* sel,
                                                       ZeroSpan zero, StampOps times) {
  put_stamp(times.stamp);
  put_stamp(times.stamp2);
  if (times.keep_from) {  // one of the times cleared below
    if (blockIdx.x == 0 && threadIdx.x == 0) *times.keep_to = *times.keep_from;
    __syncthreads();
  }
  clear_stamps(times.clear);
  const uint32_t tid = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
  for (uint32_t i = tid; i < zero.n; i += stride) zero.p[i] = 0u;
  auto copy = [&](const void* src, void* dst, uint32_t bytes) {
    for (uint32_t i = tid; i < bytes / 4u; i += stride)
      static_cast<uint32_t*>(dst)[i] = static_cast<const uint32_t*>(src)[i];
  };
  copy(pack.ftc, ftc, pack.n_ftc * uint32_t(sizeof(FtcJob)));
  if (pack.n_sel) {
    copy(&pack.hsum, hsum, uint32_t(sizeof(HsumJob)));
    copy(pack.sel, sel, pack.n_sel * uint32_t(sizeof(SelectJob)));
  }
}

hipError_t launch_put_jobs(const JobPack& pack, FtcJob* d_ftc, HsumJob* d_hsum, SelectJob* d_sel, ZeroSpan zero,
                           hipStream_t stream, const StampOps& times) {
  const uint32_t blocks = min(1u + zero.n / 1024u, 64u);
  hipLaunchKernelGGL(put_jobs_kernel, dim3(blocks), dim3(256), 0, stream, pack, d_ftc, d_hsum, d_sel, zero, times);
  return hipGetLastError();
}

// Bound by the source: pinned host memory or HBM.
__global__ __launch_bounds__(256) void copy_spectrum_kernel(const float2* __restrict__ src, float2* __restrict__ dst,
                                                            uint32_t n, uint64_t* stamp, uint64_t* end,
                                                            StampSpan clear) {
  put_stamp(stamp);
  clear_stamps(clear);
  const uint32_t step = gridDim.x * 256u;
  for (uint64_t i0 = blockIdx.x * 256u + threadIdx.x; i0 < n; i0 += 4ull * step) {
    float2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = gld2(src, size_t(min(i0 + uint64_t(u) * step, uint64_t(n - 1u))));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i0 + uint64_t(u) * step < n) dst[i0 + uint64_t(u) * step] = v[u];
  }
  if (end && blockIdx.x == gridDim.x - 1u && threadIdx.x == 0) *end = wall_clock64();
}

hipError_t launch_copy_spectrum(const float2* src, float2* dst, uint32_t n, hipStream_t stream, uint64_t* stamp,
                                uint64_t* end, StampSpan clear) {
  if (n == 0) return hipSuccess;
  const uint32_t blocks = min((n + 1023u) / 1024u, 2048u);
  copy_spectrum_kernel<<<blocks, 256, 0, stream>>>(src, dst, n, stamp, end, clear);
  return hipGetLastError();
}

__global__ void stamp_kernel(uint64_t* stamp, uint64_t* stamp2, StampSpan clear) {
  put_stamp(stamp);
  put_stamp(stamp2);
  clear_stamps(clear);
}

hipError_t launch_stamp(hipStream_t stream, uint64_t* stamp, uint64_t* stamp2, StampSpan clear) {
  stamp_kernel<<<1, 64, 0, stream>>>(stamp, stamp2, clear);
  return hipGetLastError();
}

}  // namespace fdas
