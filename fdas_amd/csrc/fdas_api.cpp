// Host runtime behind the C ABI in include/fdas.h.
//
// Mirrors the reference host class FDAS (fdas/src/host/FDAS.cpp): a context
// owns the device, two buffer sets A/B with their own stream, the resident
// template spectra, the FOP and the candidate buffers.  Where the reference
// sequences ~40 OpenCL kernels over on-chip channels, one set here runs seven
// HIP kernels in order on its stream: spectrum copy, job descriptors, fused FT
// convolution, harmonic summing with thresholding, and per-plane selection
// (histogram, compaction, final).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <cmath>
#include <complex>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "fdas_geometry.h"
#include "fdas_host.h"
#include "fdas_jobs.h"
#include "fdas_kernels.h"
#include "fdas_plan.h"

using namespace fdas;

namespace {

constexpr uint32_t kMaxFtcJobs = 64;  // row groups per FT-convolution launch

// Device times of a launch (clock ticks, in pinned host memory, 0: not taken): START, INPUT (spectrum in place),
// FTC_K (FT-convolution kernel start), FTC (its end where no summing follows at once), HSUM_K0 (harmonic-summing
// kernel start), HSUM_K1 (selection start), then the end of each plane's selection.  TAKEN is no time of its own: the
// kernel after a staged spectrum's copy has started, and the staging buffer may be rewritten.
enum Stamp {
  ST_START = 0, ST_INPUT, ST_FTC_K, ST_FTC, ST_HSUM_K0, ST_HSUM_K1, ST_ENDS, ST_COUNT = ST_ENDS + kMaxHarmonics,
  ST_TAKEN = ST_COUNT, ST_WORDS
};

// Host spectra up to this size are taken through pinned memory by a kernel; larger ones by a copy command.  Launch and
// wait with 5 templates, by copy command and by kernel: 74 and 44 us at 4096 bins, 73 and 62 at 32768, 109 and 93 at
// 2^17 (1 MiB), 139 and 138 at 2^18, 199 and 210 at 2^19, where the host's copy costs more than the signal saves.
constexpr size_t kStagedInput = 1 << 20;

struct DevSet {
  float2* input = nullptr;
  float2* hperm = nullptr;
  float* fop = nullptr;
  float2* tiles = nullptr;
  float* plane = nullptr;
  uint32_t* spill_key = nullptr;
  float* spill_pwr = nullptr;
  uint32_t* counts = nullptr;      // [H][kPlaneCounters]
  uint32_t* compact_key = nullptr;
  float* compact_pwr = nullptr;
  FtcJob* d_ftc = nullptr;
  HsumJob* d_hsum = nullptr;
  SelectJob* d_sel = nullptr;
  float* quant = nullptr;          // quantile thresholds: block maxima, then [4H] thresholds, counts, order statistics

  FtcJob* h_ftc = nullptr;         // pinned staging of more than kPackFtcJobs row groups
  JobPack pack;                    // the launches' job descriptors
  // The lists, in pinned host memory that the selection kernel writes (one allocation).
  uint32_t* h_out_key = nullptr;   // [H][cap]
  float* h_out_pwr = nullptr;      // [H][cap]
  uint32_t* h_out_n = nullptr;     // [H] kept entries
  uint32_t* h_counts = nullptr;    // [H] detections
  uint32_t* h_quant = nullptr;     // [4H] mirror of quant's tail

  hipStream_t stream = nullptr;
  uint64_t* h_stamp = nullptr;       // [ST_WORDS] pinned
  bool in_flight = false;            // work was enqueued since the stream was last waited for
  bool ftc_to_hsum = false;          // the summing followed the convolution at once: its start is the other's end
  float2* h_input = nullptr;         // pinned staging of small host spectra
  bool input_pending = false;        // h_input may still be read by the device
  hipEvent_t hsum_done = nullptr;    // end of the last summing kernel, where the other set is in use
  hipEvent_t staged_ftc = nullptr;   // h_ftc may be rewritten once this completes
  bool used = false;                 // a convolution has been launched
  bool hsum_recorded = false;        // hsum_done has been recorded
  bool ftc_pending = false;

  std::vector<FtcJob> ftc_plan[3];  // convolution jobs per part (empty: not planned for these templates)
  std::vector<uint32_t> row_taps;  // non-zero extent of each template row (sets per-group overlaps)
  bool templates = false;
  bool has_input = false;
  bool fop_valid = false;
  bool cands_valid = false;
  bool tiles_valid = false;
  float thr[kMaxHarmonics] = {};
  bool thr_set = false;

  bool launched = false;
  uint32_t* user_loc = nullptr;
  float* user_pwr = nullptr;
  bool delivered = false;  // the caller's arrays hold the launch's lists, the set's own hold another pass's
  uint32_t delivered_counts[kMaxHarmonics] = {};
  bool gated = false;
  fdas_part gated_part = FDAS_ALL;
  float gated_thr[kMaxHarmonics] = {};
};

}  // namespace

struct fdas_ctx {
  fdas_config cfg{};
  Geometry geo{};
  uint32_t c = 0;
  uint32_t spill = 0;
  fdas_log_fn log = nullptr;
  void* user = nullptr;
  std::string last_error;
  float2* tw1 = nullptr;
  float2* tw2 = nullptr;
  DevSet set[2];
  uint64_t epoch = 0;       // device clock at creation
  double clock_khz = 1e5;
  uint32_t n_cu = 256;
  bool sync_pipeline = false;
  // print_stats state; the reference keeps it file-static (FDAS.cpp:640-641)
  float pipeline_start = 0.f;
  float pipeline_accum = 0.f;
  unsigned pipeline_launches = 0;
};

namespace {

void emit(fdas_ctx* ctx, int level, const std::string& msg) {
  if (ctx && ctx->log) ctx->log(level, msg.c_str(), ctx->user);
}

fdas_status fail(fdas_ctx* ctx, fdas_status st, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  if (ctx) {
    ctx->last_error = std::string("[ERROR] ") + buf;
    emit(ctx, FDAS_LOG_ERROR, ctx->last_error);
  }
  return st;
}

void info(fdas_ctx* ctx, const char* fmt, ...) {
  if (!ctx || !ctx->log) return;
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  emit(ctx, FDAS_LOG_INFO, std::string("[INFO] ") + buf);
}

#define HIPCK(ctx, expr)                                                                                       \
  do {                                                                                                         \
    hipError_t e_ = (expr);                                                                                    \
    if (e_ != hipSuccess)                                                                                      \
      return fail(ctx, FDAS_EDEVICE, "HIP call failed with status %d (%s):\n          %s [%s:%d]", int(e_), \
                  hipGetErrorString(e_), #expr, __FILE__, __LINE__);                                           \
  } while (0)

#define CHECK_SET(ctx, set)                                                      \
  do {                                                                           \
    if (!(ctx)) return FDAS_EINVAL;                                              \
    if ((set) != FDAS_SET_A && (set) != FDAS_SET_B)                              \
      return fail(ctx, FDAS_EINVAL, "invalid buffer set %d", int(set));          \
  } while (0)

bool valid_part(fdas_part p) { return p == FDAS_NEGATIVE || p == FDAS_POSITIVE || p == FDAS_ALL; }

void part_rows(const fdas_ctx* ctx, fdas_part p, uint32_t* begin, uint32_t* count) {
  switch (p) {
    case FDAS_NEGATIVE: *begin = 0; *count = ctx->c + 1; break;
    case FDAS_POSITIVE: *begin = ctx->c; *count = ctx->c + 1; break;
    default: *begin = 0; *count = ctx->cfg.n_templates; break;
  }
}

template <typename T>
fdas_status dev_alloc(fdas_ctx* ctx, T** p, size_t count) {
  *p = nullptr;
  if (count == 0) return FDAS_OK;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(p), count * sizeof(T));
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
    return fail(ctx, FDAS_ENOMEM, "device allocation of %zu bytes failed (%s)", count * sizeof(T),
                hipGetErrorString(e));
  }
  return FDAS_OK;
}

template <typename T>
fdas_status host_alloc(fdas_ctx* ctx, T** p, size_t count, unsigned flags = 0) {
  *p = nullptr;
  hipError_t e = hipHostMalloc(reinterpret_cast<void**>(p), std::max<size_t>(count, 1) * sizeof(T), flags);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    *p = nullptr;
    return fail(ctx, FDAS_ENOMEM, "pinned host allocation of %zu bytes failed (%s)", count * sizeof(T),
                hipGetErrorString(e));
  }
  return FDAS_OK;
}

// Wait until a host job staging buffer may be rewritten (its last copy to the device is done).
fdas_status wait_staging(fdas_ctx* ctx, hipEvent_t ev, bool& pending) {
  if (pending) {
    HIPCK(ctx, hipEventSynchronize(ev));
    pending = false;
  }
  return FDAS_OK;
}

void clear_stamps(DevSet& s, int from, int to) {
  for (int i = from; i <= to; ++i) reinterpret_cast<volatile uint64_t*>(s.h_stamp)[i] = 0;
}

StampSpan stamp_span(const DevSet& s, int from, int to) { return {s.h_stamp + from, uint32_t(to - from + 1)}; }

// The times from .. to are about to be taken anew.  An idle set's read as not taken from now on; kernels of an
// earlier sequence may still write them otherwise, and the new sequence's first kernel clears them.
void renew_stamps(DevSet& s, int from, int to) {
  if (!s.in_flight) clear_stamps(s, from, to);
  s.in_flight = true;
}

fdas_status stamp(fdas_ctx* ctx, DevSet& s, Stamp at) {
  HIPCK(ctx, launch_stamp(s.stream, s.h_stamp + at));
  return FDAS_OK;
}

// The clock at a stamp (ST_ENDS: the last plane's), 0 where it was not taken.
uint64_t clock_at(const fdas_ctx* ctx, const DevSet& s, int at) {
  const volatile uint64_t* t = s.h_stamp;
  if (at == ST_FTC && s.ftc_to_hsum) at = ST_HSUM_K0;
  if (at != ST_ENDS) return t[at];
  uint64_t last = 0;
  for (uint32_t p = 0; p < ctx->cfg.n_harmonics; ++p) {
    const uint64_t v = t[ST_ENDS + p];
    if (v == 0) return 0;
    last = std::max(last, v);
  }
  return last;
}

float elapsed(const fdas_ctx* ctx, const DevSet& s, int a, int b) {
  const uint64_t ta = clock_at(ctx, s, a), tb = clock_at(ctx, s, b);
  return ta && tb > ta ? float(double(tb - ta) / ctx->clock_khz) : 0.f;
}

// Milliseconds since creation, 0 where the stamp was not taken.
float since_epoch(const fdas_ctx* ctx, const DevSet& s, int at) {
  const uint64_t t = clock_at(ctx, s, at);
  return t > ctx->epoch ? float(double(t - ctx->epoch) / ctx->clock_khz) : 0.f;
}

// Waits for the set's stream: lists and stamps are in host memory, the staged spectrum has been read.
fdas_status drain(fdas_ctx* ctx, DevSet& s) {
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  s.input_pending = s.in_flight = false;
  return FDAS_OK;
}

// Waits until the device has read the staged spectrum, not for the work behind it: a launch over one that was not
// waited for is enqueued while that one runs.
fdas_status wait_taken(fdas_ctx* ctx, DevSet& s) {
  const volatile uint64_t* taken = s.h_stamp + ST_TAKEN;
  for (uint32_t spin = 1; s.input_pending && !*taken; ++spin) {
    if (spin % 256 != 0) continue;
    const hipError_t e = hipStreamQuery(s.stream);  // idle: whatever was enqueued has run
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    HIPCK(ctx, e);
    break;
  }
  s.input_pending = false;
  return FDAS_OK;
}

// The convolution jobs of the part.  Planned once per part and template bank: the
// row grouping (a dynamic program over the rows, about 35 us on the host for 85) depends on
// nothing else that changes between launches.
const std::vector<FtcJob>& ftc_jobs(const fdas_ctx* ctx, DevSet& s, fdas_part part) {
  std::vector<FtcJob>& jobs = s.ftc_plan[part];
  if (!jobs.empty()) return jobs;
  uint32_t rb, nr;
  part_rows(ctx, part, &rb, &nr);
  jobs = plan_ftc_rows(ctx->cfg.tile, ctx->geo.n_bins, ctx->cfg.max_taps, s.row_taps, rb, nr, kMaxFtcJobs);
  fit_ftc_items(jobs, ftconv_slots(ctx->cfg.tile, ctx->n_cu));
  uint32_t item = 0;
  for (FtcJob& j : jobs) {
    j.spectrum = s.input;
    j.fop = s.fop;
    j.hperm = s.hperm;
    j.item_begin = item;
    item += j.n_tiles * j.n_chunks;
  }
  return jobs;
}

// The convolution jobs of the part into the pack (or, beyond its size, the pinned staging array).
// Returns the work items; *n_jobs = jobs.
fdas_status fill_ftc(fdas_ctx* ctx, DevSet& s, fdas_part part, uint32_t* n_jobs, uint32_t* n_items) {
  const std::vector<FtcJob>& jobs = ftc_jobs(ctx, s, part);
  *n_jobs = uint32_t(jobs.size());
  *n_items = jobs.back().item_begin + jobs.back().n_tiles * jobs.back().n_chunks;
  s.pack.n_ftc = 0;
  if (jobs.size() <= kPackFtcJobs) {
    std::copy(jobs.begin(), jobs.end(), s.pack.ftc);
    s.pack.n_ftc = *n_jobs;
    return FDAS_OK;
  }
  const fdas_status st = wait_staging(ctx, s.staged_ftc, s.ftc_pending);
  if (st != FDAS_OK) return st;
  std::copy(jobs.begin(), jobs.end(), s.h_ftc);
  HIPCK(ctx, hipMemcpyAsync(s.d_ftc, s.h_ftc, sizeof(FtcJob) * jobs.size(), hipMemcpyHostToDevice, s.stream));
  HIPCK(ctx, hipEventRecord(s.staged_ftc, s.stream));
  s.ftc_pending = true;
  return FDAS_OK;
}

// The summing and selection jobs of a pass over the part into the pack.
void fill_hsum(fdas_ctx* ctx, DevSet& s, fdas_part part, const float* thr) {
  uint32_t rb, nr;
  part_rows(ctx, part, &rb, &nr);
  const uint32_t H = ctx->cfg.n_harmonics;
  HsumJob& j = s.pack.hsum;
  j = HsumJob{};
  j.fop = s.fop;
  j.n_bins = ctx->geo.n_bins;
  j.n_templates = ctx->cfg.n_templates;
  j.row_begin = rb;
  j.n_rows = nr;
  j.n_harmonics = H;
  j.spill_cap = ctx->spill;
  j.block_begin = 0;
  hsum_row_chunks(nr, &j.rows_per_block, &j.n_row_chunks, hsum_rows_for(j.n_bins, nr));
  j.spill_key = s.spill_key;
  j.spill_pwr = s.spill_pwr;
  j.counts = s.counts;
  for (uint32_t k = 0; k < H; ++k) j.thr[k] = thr[k];
  const uint32_t cap = ctx->cfg.cands_per_harmonic, ccap = cap + kSelectPool;
  for (uint32_t p = 0; p < H; ++p) {
    SelectJob& q = s.pack.sel[p];
    q.spill_key = s.spill_key + size_t(p) * ctx->spill;
    q.spill_pwr = s.spill_pwr + size_t(p) * ctx->spill;
    q.count = s.counts + size_t(p) * kPlaneCounters;
    q.spill_cap = ctx->spill;
    q.cap = cap;
    q.thr = thr[p];
    q.compact_cap = ccap;
    q.hist = s.counts + size_t(p) * kPlaneCounters + 2;
    q.compact_key = s.compact_key + size_t(p) * ccap;
    q.compact_pwr = s.compact_pwr + size_t(p) * ccap;
    q.compact_n = s.counts + size_t(p) * kPlaneCounters + 1;
    q.out_key = s.h_out_key + size_t(p) * cap;
    q.out_pwr = s.h_out_pwr + size_t(p) * cap;
    q.out_n = s.h_out_n + p;
    q.out_count = s.h_counts + p;
  }
  s.pack.n_sel = H;
}

// Takes the pack's jobs to the device, with the counters cleared when a summing pass is among them.
fdas_status put_jobs(fdas_ctx* ctx, DevSet& s, const StampOps& times = StampOps{}) {
  ZeroSpan zero;
  if (s.pack.n_sel) zero = {s.counts, ctx->cfg.n_harmonics * kPlaneCounters};
  HIPCK(ctx, launch_put_jobs(s.pack, s.d_ftc, s.d_hsum, s.d_sel, zero, s.stream, times));
  s.pack.n_ftc = s.pack.n_sel = 0;
  return FDAS_OK;
}

fdas_status run_ftc(fdas_ctx* ctx, DevSet& s, uint32_t n_jobs, uint32_t n_items) {
  // The two sets' kernels take turns: this convolution starts once the other
  // set's last summing kernel has finished (both kinds of kernel are VALU-bound,
  // and side by side they only slow each other down), while that set's
  // selection, and this set's input copy, still overlap.
  const DevSet& other = &s == &ctx->set[0] ? ctx->set[1] : ctx->set[0];
  if (other.hsum_recorded) HIPCK(ctx, hipStreamWaitEvent(s.stream, other.hsum_done, 0));
  s.used = true;
  HIPCK(ctx, launch_ftconv(int(ctx->cfg.tile), s.d_ftc, n_jobs, n_items, ctx->tw1, ctx->tw2, n_items, s.stream,
                           s.h_stamp + ST_FTC_K));
  return FDAS_OK;
}

// The summing and selection kernels of the jobs on the device.
fdas_status run_hsum(fdas_ctx* ctx, DevSet& s) {
  const uint32_t H = ctx->cfg.n_harmonics;
  const HsumJob& j = s.pack.hsum;
  const uint32_t blocks = (ctx->geo.n_bins + kHsumBinsPerBlock - 1) / kHsumBinsPerBlock * j.n_row_chunks;
  HIPCK(ctx, launch_hsum(s.d_hsum, 1, blocks, H, s.stream, s.h_stamp + ST_HSUM_K0));
  const DevSet& other = &s == &ctx->set[0] ? ctx->set[1] : ctx->set[0];
  if (other.used) {  // its next convolution waits for this summing
    HIPCK(ctx, hipEventRecord(s.hsum_done, s.stream));
    s.hsum_recorded = true;
  }
  HIPCK(ctx, launch_select(s.d_sel, H, ctx->cfg.cands_per_harmonic, s.stream, s.h_stamp + ST_HSUM_K1,
                           s.h_stamp + ST_ENDS));
  return FDAS_OK;
}

// Times of a sequence that begins with a convolution and ends at `last`.  start: it starts here (no input step
// before it).
StampOps ftc_stamps(DevSet& s, bool start, int last) {
  renew_stamps(s, start ? ST_START : ST_INPUT, last);
  StampOps t;
  t.stamp = s.h_stamp + ST_INPUT;
  t.stamp2 = s.h_stamp + (start ? ST_START : ST_TAKEN);
  t.clear = stamp_span(s, ST_FTC_K, last);
  return t;
}

// Convolution alone.
fdas_status enqueue_ftc(fdas_ctx* ctx, DevSet& s, fdas_part part, bool start) {
  const StampOps times = ftc_stamps(s, start, ST_FTC);
  s.ftc_to_hsum = false;
  uint32_t n_jobs, n_items;
  fdas_status st = fill_ftc(ctx, s, part, &n_jobs, &n_items);
  if (st != FDAS_OK) return st;
  // (with no jobs in the pack the kernel sees to the times only)
  if ((st = put_jobs(ctx, s, times)) != FDAS_OK) return st;
  if ((st = run_ftc(ctx, s, n_jobs, n_items)) != FDAS_OK) return st;
  return stamp(ctx, s, ST_FTC);
}

// Times of a summing pass on its own: the convolution's end is kept, the pass's are not taken yet.
StampOps hsum_stamps(DevSet& s) {
  StampOps t;
  if (s.ftc_to_hsum && s.in_flight) {
    t.keep_from = s.h_stamp + ST_HSUM_K0;
    t.keep_to = s.h_stamp + ST_FTC;
  } else if (s.ftc_to_hsum) {
    s.h_stamp[ST_FTC] = s.h_stamp[ST_HSUM_K0];
  }
  s.ftc_to_hsum = false;
  renew_stamps(s, ST_HSUM_K0, ST_COUNT - 1);
  t.clear = stamp_span(s, ST_HSUM_K0, ST_COUNT - 1);
  return t;
}

fdas_status enqueue_hsum(fdas_ctx* ctx, DevSet& s, fdas_part part, const float* thr) {
  const StampOps times = hsum_stamps(s);
  fill_hsum(ctx, s, part, thr);
  const fdas_status st = put_jobs(ctx, s, times);
  return st == FDAS_OK ? run_hsum(ctx, s) : st;
}

// Convolution and summing of one launch, their jobs taken to the device together.
fdas_status enqueue_search(fdas_ctx* ctx, DevSet& s, fdas_part part, const float* thr, bool start) {
  const StampOps times = ftc_stamps(s, start, ST_COUNT - 1);
  s.ftc_to_hsum = true;
  uint32_t n_jobs, n_items;
  fdas_status st = fill_ftc(ctx, s, part, &n_jobs, &n_items);
  if (st != FDAS_OK) return st;
  fill_hsum(ctx, s, part, thr);
  if ((st = put_jobs(ctx, s, times)) != FDAS_OK) return st;
  if ((st = run_ftc(ctx, s, n_jobs, n_items)) != FDAS_OK) return st;
  return run_hsum(ctx, s);
}

// Converts the staged lists to the reference's 32-bit layout (gen_info.h:62-73).
void to_reference_lists(const fdas_ctx* ctx, const DevSet& s, uint32_t* loc, float* pwr) {
  const uint32_t H = ctx->cfg.n_harmonics, cap = ctx->cfg.cands_per_harmonic;
  const int c = int(ctx->c);
  const uint32_t inv = invalid_location(c);
  for (uint32_t p = 0; p < H; ++p) {
    const uint32_t n = std::min(s.h_out_n[p], cap);
    for (uint32_t i = 0; i < cap; ++i) {
      const size_t o = size_t(p) * cap + i;
      if (i < n) {
        const uint32_t key = s.h_out_key[o];
        const int row = int(key >> kKeyBinBits);
        const uint32_t bin = key & ((1u << kKeyBinBits) - 1);
        loc[o] = encode_location(p + 1, row - c, bin, c);
        pwr[o] = s.h_out_pwr[o];
      } else {
        loc[o] = inv;
        pwr[o] = -1.0f;
      }
    }
  }
}

bool reference_format_ok(const fdas_ctx* ctx) { return ctx->cfg.n_templates <= 127 && ctx->cfg.n_harmonics <= 8; }

// counts: [H] detections
fdas_status overflow_status(fdas_ctx* ctx, const uint32_t* counts) {
  for (uint32_t p = 0; p < ctx->cfg.n_harmonics; ++p)
    if (counts[p] > ctx->spill)
      return fail(ctx, FDAS_EOVERFLOW,
                  "plane %u: %u detections exceed the spill capacity %u; lists are incomplete (raise the "
                  "threshold or spill_per_harmonic)",
                  p + 1, counts[p], ctx->spill);
  return FDAS_OK;
}

// The finished launch's lists to the caller's arrays before another pass overwrites the set's.
void deliver_early(const fdas_ctx* ctx, DevSet& s) {
  to_reference_lists(ctx, s, s.user_loc, s.user_pwr);
  std::copy(s.h_counts, s.h_counts + ctx->cfg.n_harmonics, s.delivered_counts);
  s.delivered = true;
}

fdas_status flush_gated(fdas_ctx* ctx, int set) {
  DevSet& s = ctx->set[set];
  if (!s.gated) return FDAS_OK;
  s.gated = false;
  return enqueue_hsum(ctx, s, s.gated_part, s.gated_thr);
}

void free_set(DevSet& s) {
  (void)hipFree(s.input);
  (void)hipFree(s.hperm);
  (void)hipFree(s.fop);
  (void)hipFree(s.tiles);
  (void)hipFree(s.plane);
  (void)hipFree(s.spill_key);
  (void)hipFree(s.spill_pwr);
  (void)hipFree(s.compact_key);
  (void)hipFree(s.compact_pwr);
  (void)hipFree(s.counts);
  (void)hipFree(s.d_ftc);
  (void)hipFree(s.d_hsum);
  (void)hipFree(s.d_sel);
  (void)hipFree(s.quant);
  (void)hipHostFree(s.h_quant);
  (void)hipHostFree(s.h_ftc);
  (void)hipHostFree(s.h_out_key);  // and h_out_pwr, h_out_n, h_counts
  if (s.hsum_done) (void)hipEventDestroy(s.hsum_done);
  (void)hipHostFree(s.h_stamp);
  (void)hipHostFree(s.h_input);
  if (s.staged_ftc) (void)hipEventDestroy(s.staged_ftc);
  if (s.stream) (void)hipStreamDestroy(s.stream);
  s = DevSet{};
}

fdas_status validate_config(fdas_ctx* ctx, const fdas_config& c) {
  if (c.n_bins == 0 || c.n_bins > kMaxBins)
    return fail(ctx, FDAS_EINVAL, "n_bins %u outside [1, %u]", c.n_bins, kMaxBins);
  if (c.n_templates == 0 || (c.n_templates & 1u) == 0 || c.n_templates > kMaxTemplates)
    return fail(ctx, FDAS_EINVAL, "n_templates %u must be odd and <= %u", c.n_templates, kMaxTemplates);
  if (c.tile != 1024 && c.tile != 2048 && c.tile != 4096)
    return fail(ctx, FDAS_EINVAL, "tile %u must be 1024, 2048 or 4096", c.tile);
  if (c.max_taps == 0 || overlap_for(c.max_taps) >= c.tile)
    return fail(ctx, FDAS_EINVAL, "max_taps %u leaves no payload in a %u-point tile", c.max_taps, c.tile);
  if (c.n_harmonics == 0 || c.n_harmonics > kMaxHarmonics)
    return fail(ctx, FDAS_EINVAL, "n_harmonics %u outside [1, %u]", c.n_harmonics, kMaxHarmonics);
  if (c.cands_per_harmonic == 0 || c.cands_per_harmonic > kSelectMaxCap)
    return fail(ctx, FDAS_EINVAL, "cands_per_harmonic %u outside [1, %u]", c.cands_per_harmonic, kSelectMaxCap);
  return FDAS_OK;
}

}  // namespace

// ---------------------------------------------------------------------------

extern "C" void fdas_default_config(fdas_config* cfg) {
  if (!cfg) return;
  *cfg = fdas_config{};
  cfg->n_bins = 0;
  cfg->n_templates = 85;
  cfg->max_taps = 421;
  cfg->tile = 2048;
  cfg->n_harmonics = 8;
  cfg->cands_per_harmonic = 512;
  cfg->spill_per_harmonic = 0;
  cfg->device = 0;
  cfg->flags = 0;
}

extern "C" const char* fdas_status_string(fdas_status s) {
  switch (s) {
    case FDAS_OK: return "ok";
    case FDAS_EINVAL: return "invalid argument";
    case FDAS_ENOMEM: return "out of memory";
    case FDAS_EDEVICE: return "device error";
    case FDAS_EUNSUPPORTED: return "unsupported";
    case FDAS_EBUSY: return "busy";
    case FDAS_ESTATE: return "call out of order";
    case FDAS_EOVERFLOW: return "candidate spill overflow";
    case FDAS_ECANCELED: return "request canceled";
  }
  return "unknown status";
}

extern "C" const char* fdas_last_error(const fdas_ctx* ctx) { return ctx ? ctx->last_error.c_str() : ""; }

extern "C" fdas_status fdas_create(const fdas_config* cfg, fdas_log_fn log, void* user, fdas_ctx** out) {
  if (!cfg || !out) return FDAS_EINVAL;
  *out = nullptr;
  fdas_ctx* ctx = new (std::nothrow) fdas_ctx();
  if (!ctx) return FDAS_ENOMEM;
  ctx->log = log;
  ctx->user = user;
  ctx->cfg = *cfg;
  fdas_status st = validate_config(ctx, ctx->cfg);
  if (st != FDAS_OK) {
    delete ctx;
    return st;
  }
  ctx->geo = make_geometry(cfg->n_bins, cfg->tile, cfg->max_taps);
  ctx->c = cfg->n_templates / 2;
  ctx->spill = cfg->spill_per_harmonic ? cfg->spill_per_harmonic : default_spill(cfg->n_templates, cfg->n_bins);
  ctx->sync_pipeline = (cfg->flags & FDAS_FLAG_SYNC_PIPELINE) != 0;

  auto bail = [&](fdas_status s) {
    for (auto& set : ctx->set) free_set(set);
    (void)hipFree(ctx->tw1);
    (void)hipFree(ctx->tw2);
    delete ctx;
    return s;
  };

  int n_dev = 0;
  hipError_t e = hipGetDeviceCount(&n_dev);
  if (e != hipSuccess || n_dev == 0) {
    fail(ctx, FDAS_EDEVICE, "no HIP device found (%s)", hipGetErrorString(e));
    return bail(FDAS_EDEVICE);
  }
  if (cfg->device < 0 || cfg->device >= n_dev) {
    fail(ctx, FDAS_EINVAL, "device %d outside [0, %d)", cfg->device, n_dev);
    return bail(FDAS_EINVAL);
  }
  if ((e = hipSetDevice(cfg->device)) != hipSuccess) {
    fail(ctx, FDAS_EDEVICE, "hipSetDevice(%d) failed (%s)", cfg->device, hipGetErrorString(e));
    return bail(FDAS_EDEVICE);
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, cfg->device) == hipSuccess)
    info(ctx, "Device[%d]: %s (%s, %d CUs)", cfg->device, prop.name, prop.gcnArchName, prop.multiProcessorCount);

  // Twiddle tables in FP64, rounded once.
  const uint32_t S = cfg->tile;
  std::vector<float2> tw1, tw2;
  make_twiddles(S, tw1, tw2);
  if ((st = dev_alloc(ctx, &ctx->tw1, tw1.size())) != FDAS_OK) return bail(st);
  if ((st = dev_alloc(ctx, &ctx->tw2, tw2.size())) != FDAS_OK) return bail(st);
  if (hipMemcpy(ctx->tw1, tw1.data(), tw1.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(ctx->tw2, tw2.data(), tw2.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess) {
    fail(ctx, FDAS_EDEVICE, "twiddle upload failed");
    return bail(FDAS_EDEVICE);
  }
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, cfg->device) == hipSuccess && khz > 0)
    ctx->clock_khz = khz;
  int n_cu = 0;
  if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, cfg->device) == hipSuccess && n_cu > 0)
    ctx->n_cu = uint32_t(n_cu);

  const size_t N = cfg->n_bins, T = cfg->n_templates, H = cfg->n_harmonics, cap = cfg->cands_per_harmonic;
  for (auto& s : ctx->set) {
    if ((st = dev_alloc(ctx, &s.input, N)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.hperm, T * S)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.fop, T * N)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.spill_key, H * ctx->spill)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.spill_pwr, H * ctx->spill)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.compact_key, H * (cap + kSelectPool))) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.compact_pwr, H * (cap + kSelectPool))) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.counts, H * kPlaneCounters)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.d_ftc, kMaxFtcJobs)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.d_hsum, 1)) != FDAS_OK) return bail(st);
    if ((st = dev_alloc(ctx, &s.d_sel, H)) != FDAS_OK) return bail(st);
    if ((st = host_alloc(ctx, &s.h_ftc, kMaxFtcJobs)) != FDAS_OK) return bail(st);
    if ((st = host_alloc(ctx, &s.h_out_key, 2 * H * cap + 2 * H, hipHostMallocCoherent)) != FDAS_OK) return bail(st);
    s.h_out_pwr = reinterpret_cast<float*>(s.h_out_key + H * cap);
    s.h_out_n = s.h_out_key + 2 * H * cap;
    s.h_counts = s.h_out_n + H;
    std::memset(s.h_out_n, 0, sizeof(uint32_t) * H);
    std::memset(s.h_counts, 0, sizeof(uint32_t) * H);
    if (hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) != hipSuccess)
      return bail(fail(ctx, FDAS_EDEVICE, "stream creation failed"));
    if ((st = host_alloc(ctx, &s.h_stamp, ST_WORDS, hipHostMallocCoherent)) != FDAS_OK) return bail(st);
    clear_stamps(s, 0, ST_COUNT - 1);
    static_assert(ST_COUNT <= 64, "cleared by one workgroup's threads");
    if (N * sizeof(float2) <= kStagedInput && (st = host_alloc(ctx, &s.h_input, N)) != FDAS_OK) return bail(st);
    if (hipEventCreateWithFlags(&s.hsum_done, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s.staged_ftc, hipEventDisableTiming) != hipSuccess)
      return bail(fail(ctx, FDAS_EDEVICE, "event creation failed"));
    // a FOP that was never written reads as zeros
    if (hipMemset(s.fop, 0, T * N * sizeof(float)) != hipSuccess ||
        hipMemset(s.counts, 0, H * kPlaneCounters * sizeof(uint32_t)) != hipSuccess)
      return bail(fail(ctx, FDAS_EDEVICE, "buffer initialisation failed"));
  }
  uint64_t* const clock = ctx->set[0].h_stamp;
  if (launch_stamp(ctx->set[0].stream, clock) != hipSuccess || hipDeviceSynchronize() != hipSuccess)
    return bail(fail(ctx, FDAS_EDEVICE, "device synchronisation failed"));
  ctx->epoch = *static_cast<volatile uint64_t*>(clock);
  *clock = 0;
  info(ctx, "Geometry: N=%u, T=%u, S=%u, overlap=%u, payload=%u, tiles=%u, H=%u, cap=%u, spill=%u", cfg->n_bins,
       cfg->n_templates, S, ctx->geo.overlap, ctx->geo.payload, ctx->geo.n_tiles, cfg->n_harmonics,
       cfg->cands_per_harmonic, ctx->spill);
  *out = ctx;
  return FDAS_OK;
}

extern "C" void fdas_destroy(fdas_ctx* ctx) {
  if (!ctx) return;
  (void)hipSetDevice(ctx->cfg.device);
  for (auto& s : ctx->set)
    if (s.stream) (void)hipStreamSynchronize(s.stream);
  for (auto& s : ctx->set) free_set(s);
  (void)hipFree(ctx->tw1);
  (void)hipFree(ctx->tw2);
  delete ctx;
}

extern "C" uint64_t fdas_get_size(const fdas_ctx* ctx, fdas_size_kind which) {
  if (!ctx) return 0;
  switch (which) {
    case FDAS_SIZE_INPUT: return ctx->geo.n_bins;
    case FDAS_SIZE_TILES: return uint64_t(ctx->geo.n_tiles) * ctx->cfg.tile;
    case FDAS_SIZE_TEMPLATES: return uint64_t(ctx->cfg.n_templates) * ctx->cfg.tile;
    case FDAS_SIZE_THRESHOLDS: return ctx->cfg.n_harmonics;
    case FDAS_SIZE_FOP: return uint64_t(ctx->cfg.n_templates) * ctx->geo.n_bins;
    case FDAS_SIZE_CANDIDATES: return uint64_t(ctx->cfg.n_harmonics) * ctx->cfg.cands_per_harmonic;
  }
  return 0;
}

static fdas_status upload_spectra(fdas_ctx* ctx, int set, const std::vector<std::complex<double>>& spec) {
  // Stored as [t][slot][tid] (kernel register order after the forward tile transform), scaled by 1/S.
  const std::vector<float2> perm = kernel_template_layout(spec, ctx->cfg.n_templates, ctx->cfg.tile);
  DevSet& s = ctx->set[set];
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  HIPCK(ctx, hipMemcpy(s.hperm, perm.data(), perm.size() * sizeof(float2), hipMemcpyHostToDevice));
  s.templates = true;
  info(ctx, "Uploaded template coefficients");
  return FDAS_OK;
}

static void set_row_taps(DevSet& s, const std::vector<uint32_t>& taps) {
  s.row_taps = taps;
  for (auto& plan : s.ftc_plan) plan.clear();
}

// Natural bin of entry i of a row stored in 4-parallel FFT order:
// stored[4m + j] = natural[bitrev2(j) * S/4 + m] (tmpl-gen.py:145-153, ft_conv.py:185-194).
static inline uint32_t p4_natural_index(uint32_t i, uint32_t S) {
  const uint32_t j = i & 3u, m = i >> 2;
  const uint32_t br = ((j & 1u) << 1) | (j >> 1);
  return br * (S / 4) + m;
}

extern "C" fdas_status fdas_upload_templates(fdas_ctx* ctx, const float* spectra_c64, int set) {
  CHECK_SET(ctx, set);
  if (!spectra_c64) return fail(ctx, FDAS_EINVAL, "null template pointer");
  // spectra do not reveal the tap extent exactly: every row uses the configured max_taps
  set_row_taps(ctx->set[set], std::vector<uint32_t>(ctx->cfg.n_templates, ctx->cfg.max_taps));
  const uint32_t S = ctx->cfg.tile, T = ctx->cfg.n_templates;
  const bool p4 = (ctx->cfg.flags & FDAS_FLAG_REFERENCE_FFT_ORDER) != 0;
  std::vector<std::complex<double>> spec(size_t(T) * S);
  for (uint32_t t = 0; t < T; ++t)
    for (uint32_t i = 0; i < S; ++i) {
      const float* v = spectra_c64 + 2 * (size_t(t) * S + i);
      const uint32_t dst = p4 ? p4_natural_index(i, S) : i;
      spec[size_t(t) * S + dst] = std::complex<double>(v[0], v[1]);
    }
  return upload_spectra(ctx, set, spec);
}

extern "C" fdas_status fdas_upload_template_taps(fdas_ctx* ctx, const float* taps_c64, uint32_t n_taps, int set) {
  CHECK_SET(ctx, set);
  if (!taps_c64 || n_taps == 0) return fail(ctx, FDAS_EINVAL, "null or empty template taps");
  const uint32_t S = ctx->cfg.tile, T = ctx->cfg.n_templates;
  // Taps beyond max_taps must be zero: the tile overlap covers max_taps - 1 samples only.
  for (uint32_t t = 0; t < T; ++t)
    for (uint32_t m = ctx->cfg.max_taps; m < n_taps; ++m) {
      const float* v = taps_c64 + 2 * (size_t(t) * n_taps + m);
      if (v[0] != 0.f || v[1] != 0.f)
        return fail(ctx, FDAS_EINVAL, "template %u has a non-zero tap %u beyond max_taps %u", t, m,
                    ctx->cfg.max_taps);
    }
  std::vector<uint32_t> extent;
  const std::vector<std::complex<double>> spec = taps_to_spectra(taps_c64, T, n_taps, ctx->cfg.max_taps, S, extent);
  fdas_status st = upload_spectra(ctx, set, spec);
  if (st == FDAS_OK) set_row_taps(ctx->set[set], extent);
  return st;
}

extern "C" fdas_status fdas_upload_thresholds(fdas_ctx* ctx, const float* thresholds, int set) {
  CHECK_SET(ctx, set);
  if (!thresholds) return fail(ctx, FDAS_EINVAL, "null thresholds");
  DevSet& s = ctx->set[set];
  for (uint32_t k = 0; k < ctx->cfg.n_harmonics; ++k) s.thr[k] = thresholds[k];
  s.thr_set = true;
  info(ctx, "Uploaded thresholds");
  return FDAS_OK;
}

// Whether this device can read the whole spectrum where it is: device memory of its own, 8-byte aligned.
static bool readable_spectrum(const fdas_ctx* ctx, const void* src, size_t bytes) {
  hipPointerAttribute_t attr{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (hipPointerGetAttributes(&attr, src) != hipSuccess ||
      hipMemGetAddressRange(&base, &size, const_cast<void*>(src)) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  const uintptr_t p = reinterpret_cast<uintptr_t>(src), b = reinterpret_cast<uintptr_t>(base);
  return attr.type == hipMemoryTypeDevice && attr.device == ctx->cfg.device && p % sizeof(float2) == 0 && p >= b &&
         size >= bytes && p - b <= size - bytes;
}

// The spectrum into the set's buffer.  By a kernel, which the next one follows within 2 us, where it can be read:
// device memory, and host memory up to kStagedInput after a copy to pinned memory, as the runtime also makes one; a
// copy command's completion signal takes about 10 us to let the next kernel start.  A launch over one that was not
// waited for takes 55 us of the host at 131,072 bins (130 when it waited for all of that one's kernels); a third one
// waits until the second one's copy, behind the first one's kernels, has run.
static fdas_status upload_input(fdas_ctx* ctx, DevSet& s, const void* src, hipMemcpyKind kind) {
  const size_t bytes = sizeof(float2) * ctx->geo.n_bins;
  fdas_status st;
  if (s.input_pending && (st = wait_taken(ctx, s)) != FDAS_OK) return st;
  renew_stamps(s, 0, ST_COUNT - 1);
  s.ftc_to_hsum = false;
  const float2* from = nullptr;
  if (kind == hipMemcpyHostToDevice && s.h_input) {
    std::memcpy(s.h_input, src, bytes);
    *static_cast<volatile uint64_t*>(s.h_stamp + ST_TAKEN) = 0;
    s.input_pending = true;
    from = s.h_input;
  } else if (kind == hipMemcpyDeviceToDevice && readable_spectrum(ctx, src, bytes)) {
    from = static_cast<const float2*>(src);
  }
  if (from) {
    HIPCK(ctx, launch_copy_spectrum(from, s.input, ctx->geo.n_bins, s.stream, s.h_stamp + ST_START,
                                    s.h_stamp + ST_INPUT, stamp_span(s, ST_FTC_K, ST_COUNT - 1)));
  } else {
    HIPCK(ctx, launch_stamp(s.stream, s.h_stamp + ST_START, nullptr, stamp_span(s, ST_INPUT, ST_COUNT - 1)));
    HIPCK(ctx, hipMemcpyAsync(s.input, src, bytes, kind, s.stream));
  }
  s.has_input = true;
  s.fop_valid = false;
  s.cands_valid = false;
  s.tiles_valid = false;
  return FDAS_OK;
}

extern "C" fdas_status fdas_perform_input_tiling(fdas_ctx* ctx, const float* spectrum_c64, int set) {
  CHECK_SET(ctx, set);
  if (!spectrum_c64) return fail(ctx, FDAS_EINVAL, "null spectrum");
  DevSet& s = ctx->set[set];
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  if (!s.tiles && (st = dev_alloc(ctx, &s.tiles, size_t(ctx->geo.n_tiles) * ctx->cfg.tile)) != FDAS_OK) return st;
  if ((st = upload_input(ctx, s, spectrum_c64, hipMemcpyHostToDevice)) != FDAS_OK) return st;
  HIPCK(ctx, launch_tiles(int(ctx->cfg.tile), s.input, ctx->geo.n_bins, ctx->geo.overlap, ctx->geo.payload,
                          ctx->geo.n_tiles, ctx->tw1, ctx->tw2, s.tiles, s.stream));
  if ((st = stamp(ctx, s, ST_INPUT)) != FDAS_OK) return st;
  if ((st = drain(ctx, s)) != FDAS_OK) return st;
  s.tiles_valid = true;
  info(ctx, "Preparation duration: %.3f ms", double(elapsed(ctx, s, ST_START, ST_INPUT)));
  return FDAS_OK;
}

extern "C" fdas_status fdas_set_input_device(fdas_ctx* ctx, const void* d_spectrum_c64, int set) {
  CHECK_SET(ctx, set);
  if (!d_spectrum_c64) return fail(ctx, FDAS_EINVAL, "null device spectrum");
  DevSet& s = ctx->set[set];
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  return upload_input(ctx, s, d_spectrum_c64, hipMemcpyDeviceToDevice);
}

static fdas_status check_ready_ftc(fdas_ctx* ctx, const DevSet& s, fdas_part part) {
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  if (!s.templates) return fail(ctx, FDAS_ESTATE, "templates not uploaded for this buffer set");
  if (!s.has_input) return fail(ctx, FDAS_ESTATE, "no input spectrum in this buffer set");
  return FDAS_OK;
}

extern "C" fdas_status fdas_perform_ft_convolution(fdas_ctx* ctx, fdas_part part, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  fdas_status st = check_ready_ftc(ctx, s, part);
  if (st != FDAS_OK) return st;
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  if ((st = enqueue_ftc(ctx, s, part, false)) != FDAS_OK) return st;
  if ((st = drain(ctx, s)) != FDAS_OK) return st;
  s.fop_valid = true;
  s.cands_valid = false;
  info(ctx, "FT convolution and IFFT duration: %.3f ms", double(elapsed(ctx, s, ST_FTC_K, ST_FTC)));
  return FDAS_OK;
}

static const float* pick_thresholds(fdas_ctx* ctx, const DevSet& s, const float* thr) {
  if (thr) return thr;
  if (s.thr_set) return s.thr;
  fail(ctx, FDAS_ESTATE, "no thresholds given or uploaded");
  return nullptr;
}

extern "C" fdas_status fdas_perform_harmonic_summing(fdas_ctx* ctx, const float* thresholds, fdas_part part,
                                                     int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  const float* thr = pick_thresholds(ctx, s, thresholds);
  if (!thr) return FDAS_ESTATE;
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  if ((st = enqueue_hsum(ctx, s, part, thr)) != FDAS_OK) return st;
  if ((st = drain(ctx, s)) != FDAS_OK) return st;
  s.cands_valid = true;
  s.delivered = false;
  info(ctx, "Harmonic summing duration: %.3f ms", double(elapsed(ctx, s, ST_HSUM_K0, ST_ENDS)));
  return overflow_status(ctx, s.h_counts);
}

// The work of a launch once its spectrum is on its way: convolution, and summing
// and selection unless they are held (sync pipeline).
static fdas_status enqueue_launch(fdas_ctx* ctx, DevSet& s, fdas_part part, const float* thr, uint32_t* det_loc,
                                  float* det_pwr, bool resident) {
  fdas_status st =
      ctx->sync_pipeline ? enqueue_ftc(ctx, s, part, resident) : enqueue_search(ctx, s, part, thr, resident);
  if (st != FDAS_OK) return st;
  s.launched = true;
  s.delivered = false;
  s.user_loc = det_loc;
  s.user_pwr = det_pwr;
  if (ctx->sync_pipeline) {
    s.gated = true;
    s.gated_part = part;
    for (uint32_t k = 0; k < ctx->cfg.n_harmonics; ++k) s.gated_thr[k] = thr[k];
  }
  return FDAS_OK;
}

extern "C" fdas_status fdas_launch(fdas_ctx* ctx, const float* spectrum_c64, const float* thresholds, uint32_t* det_loc,
                                   float* det_pwr, fdas_part part, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!spectrum_c64 || !det_loc || !det_pwr) return fail(ctx, FDAS_EINVAL, "null launch argument");
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  if (!reference_format_ok(ctx))
    return fail(ctx, FDAS_EUNSUPPORTED, "T=%u/H=%u do not fit the 32-bit candidate layout; use the wide API",
                ctx->cfg.n_templates, ctx->cfg.n_harmonics);
  if (!s.templates) return fail(ctx, FDAS_ESTATE, "templates not uploaded for this buffer set");
  const float* thr = pick_thresholds(ctx, s, thresholds);
  if (!thr) return FDAS_ESTATE;
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  // Releases the other set's held harmonic summing (FDAS.cpp:549-550).
  if (ctx->sync_pipeline && (st = flush_gated(ctx, 1 - set)) != FDAS_OK) return st;
  if (s.gated && (st = flush_gated(ctx, set)) != FDAS_OK) return st;
  if ((st = upload_input(ctx, s, spectrum_c64, hipMemcpyHostToDevice)) != FDAS_OK) return st;
  return enqueue_launch(ctx, s, part, thr, det_loc, det_pwr, false);
}

extern "C" fdas_status fdas_launch_resident(fdas_ctx* ctx, const float* thresholds, uint32_t* det_loc,
                                            float* det_pwr, fdas_part part, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!det_loc || !det_pwr) return fail(ctx, FDAS_EINVAL, "null launch argument");
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  if (!reference_format_ok(ctx))
    return fail(ctx, FDAS_EUNSUPPORTED, "T=%u/H=%u do not fit the 32-bit candidate layout; use the wide API",
                ctx->cfg.n_templates, ctx->cfg.n_harmonics);
  if (!s.templates) return fail(ctx, FDAS_ESTATE, "templates not uploaded for this buffer set");
  if (!s.has_input) return fail(ctx, FDAS_ESTATE, "no input spectrum in this buffer set");
  const float* thr = pick_thresholds(ctx, s, thresholds);
  if (!thr) return FDAS_ESTATE;
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  if (ctx->sync_pipeline && (st = flush_gated(ctx, 1 - set)) != FDAS_OK) return st;
  if (s.gated && (st = flush_gated(ctx, set)) != FDAS_OK) return st;
  return enqueue_launch(ctx, s, part, thr, det_loc, det_pwr, true);
}

extern "C" fdas_status fdas_wait(fdas_ctx* ctx, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!s.launched) return fail(ctx, FDAS_ESTATE, "wait on a buffer set without a launch");
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  if (s.gated && (st = flush_gated(ctx, set)) != FDAS_OK) return st;
  if ((st = drain(ctx, s)) != FDAS_OK) return st;
  s.launched = false;
  s.fop_valid = true;
  s.cands_valid = true;
  if (s.delivered) return overflow_status(ctx, s.delivered_counts);
  to_reference_lists(ctx, s, s.user_loc, s.user_pwr);
  return overflow_status(ctx, s.h_counts);
}

extern "C" fdas_status fdas_end_pipeline(fdas_ctx* ctx, int set) {
  CHECK_SET(ctx, set);
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  return flush_gated(ctx, 1 - set);
}

extern "C" fdas_status fdas_retrieve_tiles(fdas_ctx* ctx, float* tiles_c64, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!tiles_c64) return fail(ctx, FDAS_EINVAL, "null tiles pointer");
  if (!s.tiles_valid) return fail(ctx, FDAS_ESTATE, "tiles not materialised (call perform_input_tiling)");
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  const size_t n = size_t(ctx->geo.n_tiles) * ctx->cfg.tile;
  const bool p4 = (ctx->cfg.flags & FDAS_FLAG_REFERENCE_FFT_ORDER) != 0;
  if (!p4) {
    HIPCK(ctx, hipMemcpyAsync(tiles_c64, s.tiles, n * sizeof(float2), hipMemcpyDeviceToHost, s.stream));
    HIPCK(ctx, hipStreamSynchronize(s.stream));
    return FDAS_OK;
  }
  std::vector<float2> nat(n);
  HIPCK(ctx, hipMemcpyAsync(nat.data(), s.tiles, n * sizeof(float2), hipMemcpyDeviceToHost, s.stream));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  const uint32_t S = ctx->cfg.tile;
  for (size_t t = 0; t < ctx->geo.n_tiles; ++t)
    for (uint32_t i = 0; i < S; ++i) {
      const float2 v = nat[t * S + p4_natural_index(i, S)];
      tiles_c64[2 * (t * S + i)] = v.x;
      tiles_c64[2 * (t * S + i) + 1] = v.y;
    }
  return FDAS_OK;
}

extern "C" fdas_status fdas_retrieve_fop(fdas_ctx* ctx, float* fop, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!fop) return fail(ctx, FDAS_EINVAL, "null FOP pointer");
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  const size_t n = size_t(ctx->cfg.n_templates) * ctx->geo.n_bins;
  HIPCK(ctx, hipMemcpyAsync(fop, s.fop, n * sizeof(float), hipMemcpyDeviceToHost, s.stream));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  return FDAS_OK;
}

extern "C" fdas_status fdas_inject_fop(fdas_ctx* ctx, const float* fop, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!fop) return fail(ctx, FDAS_EINVAL, "null FOP pointer");
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  const size_t n = size_t(ctx->cfg.n_templates) * ctx->geo.n_bins;
  fdas_status st;
  renew_stamps(s, ST_START, ST_FTC);
  s.ftc_to_hsum = false;
  HIPCK(ctx, launch_stamp(s.stream, s.h_stamp + ST_START, s.h_stamp + ST_INPUT, stamp_span(s, ST_FTC_K, ST_FTC)));
  HIPCK(ctx, hipMemcpyAsync(s.fop, fop, n * sizeof(float), hipMemcpyHostToDevice, s.stream));
  if ((st = stamp(ctx, s, ST_FTC)) != FDAS_OK) return st;
  s.fop_valid = true;
  s.cands_valid = false;
  return FDAS_OK;
}

extern "C" fdas_status fdas_retrieve_candidates(fdas_ctx* ctx, uint32_t* det_loc, float* det_pwr, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!det_loc || !det_pwr) return fail(ctx, FDAS_EINVAL, "null candidate pointer");
  if (!reference_format_ok(ctx))
    return fail(ctx, FDAS_EUNSUPPORTED, "T=%u/H=%u do not fit the 32-bit candidate layout; use the wide API",
                ctx->cfg.n_templates, ctx->cfg.n_harmonics);
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  to_reference_lists(ctx, s, det_loc, det_pwr);
  return FDAS_OK;
}

extern "C" fdas_status fdas_retrieve_candidates_wide(fdas_ctx* ctx, fdas_candidate* out, uint32_t capacity,
                                                     uint32_t* n_written, uint32_t* n_detected, int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!out && capacity) return fail(ctx, FDAS_EINVAL, "null candidate pointer");
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  const uint32_t H = ctx->cfg.n_harmonics, cap = ctx->cfg.cands_per_harmonic;
  const int c = int(ctx->c);
  uint32_t w = 0;
  for (uint32_t p = 0; p < H; ++p) {
    if (n_detected) n_detected[p] = s.h_counts[p];
    const uint32_t n = std::min(s.h_out_n[p], cap);
    for (uint32_t i = 0; i < n && w < capacity; ++i, ++w) {
      const uint32_t key = s.h_out_key[size_t(p) * cap + i];
      out[w].harmonic = p + 1;
      out[w].template_num = int(key >> kKeyBinBits) - c;
      out[w].bin = key & ((1u << kKeyBinBits) - 1);
      out[w].power = s.h_out_pwr[size_t(p) * cap + i];
    }
  }
  if (n_written) *n_written = w;
  return overflow_status(ctx, s.h_counts);
}

extern "C" fdas_status fdas_retrieve_harmonic_plane(fdas_ctx* ctx, uint32_t k, float* plane, fdas_part part,
                                                    int set) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!plane) return fail(ctx, FDAS_EINVAL, "null plane pointer");
  if (k == 0 || k > ctx->cfg.n_harmonics) return fail(ctx, FDAS_EINVAL, "harmonic %u outside [1, %u]", k,
                                                      ctx->cfg.n_harmonics);
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  const size_t n = size_t(ctx->cfg.n_templates) * ctx->geo.n_bins;
  fdas_status st;
  if (!s.plane && (st = dev_alloc(ctx, &s.plane, n)) != FDAS_OK) return st;
  uint32_t rb, nr;
  part_rows(ctx, part, &rb, &nr);
  HIPCK(ctx, launch_hplane(s.fop, ctx->geo.n_bins, ctx->cfg.n_templates, rb, nr, k, s.plane, s.stream));
  HIPCK(ctx, hipMemcpyAsync(plane + size_t(rb) * ctx->geo.n_bins, s.plane + size_t(rb) * ctx->geo.n_bins,
                            size_t(nr) * ctx->geo.n_bins * sizeof(float), hipMemcpyDeviceToHost, s.stream));
  HIPCK(ctx, hipStreamSynchronize(s.stream));
  return FDAS_OK;
}

// hsum.py:125-131, the "mock-up" thresholds: thr_k = quantile(HP_k, 1 - n / M)
// over the M = rows * N values of the part, linear interpolation between the
// order statistics around q (M - 1), in FP64, rounded once to float32.  The two
// order statistics are the (n+1)-th and n-th largest values.  Instead of
// sorting M values: the (n+2)-th largest block maximum B_k bounds them from
// below (n+2 blocks hold a value >= B_k), so one summing pass with a threshold
// just below B_k spills every value >= B_k, and the two are found among those.
// All of that runs on the device with one read-back; only planes with fewer
// blocks than that, or more spilled values than the lists hold, bring the host
// in, which bisects their thresholds.
extern "C" fdas_status fdas_quantile_thresholds(fdas_ctx* ctx, uint32_t n_per_plane, fdas_part part, int set,
                                                float* thresholds) {
  CHECK_SET(ctx, set);
  DevSet& s = ctx->set[set];
  if (!thresholds) return fail(ctx, FDAS_EINVAL, "null thresholds pointer");
  if (!valid_part(part)) return fail(ctx, FDAS_EINVAL, "invalid FOP part %d", int(part));
  if (!s.fop_valid) return fail(ctx, FDAS_ESTATE, "no FOP in this buffer set (run the FT convolution first)");
  uint32_t rb, nr;
  part_rows(ctx, part, &rb, &nr);
  const uint32_t N = ctx->geo.n_bins, H = ctx->cfg.n_harmonics;
  const uint64_t M = uint64_t(nr) * N;
  if (n_per_plane < 1 || n_per_plane >= M)
    return fail(ctx, FDAS_EINVAL, "candidates per plane %u outside 1 .. %llu", n_per_plane,
                (unsigned long long)(M - 1));
  HIPCK(ctx, hipSetDevice(ctx->cfg.device));
  fdas_status st;
  const size_t most = size_t(H) * hmax_blocks(N, ctx->cfg.n_templates);
  if (!s.quant && (st = dev_alloc(ctx, &s.quant, most + 4 * H)) != FDAS_OK) return st;
  if (!s.h_quant && (st = host_alloc(ctx, &s.h_quant, 4 * H)) != FDAS_OK) return st;
  float* d_thr = s.quant + most;                                  // [H] bounds
  uint32_t* d_rank = reinterpret_cast<uint32_t*>(d_thr + H);      // [3H] counts, order statistics
  const float* h_thr = reinterpret_cast<const float*>(s.h_quant);
  const uint32_t* h_rank = s.h_quant + H;
  const double q = 1.0 - double(n_per_plane) / double(M);
  const double vi = q * double(M - 1);
  const uint64_t below = uint64_t(std::floor(vi));  // ascending rank of the lower order statistic
  const double g = vi - double(below);
  // descending ranks of the two order statistics
  const uint64_t r_lo = M - 1 - below, r_hi = below + 1 < M ? M - 2 - below : r_lo;
  const uint64_t want = std::min<uint64_t>(uint64_t(n_per_plane) + 2, M);  // a spare rank for rounding
  // One summing pass over the staged jobs and the order statistics of its spill.
  auto spill_pass = [&]() -> fdas_status {
    const fdas_status r = run_hsum(ctx, s);
    if (r != FDAS_OK) return r;
    HIPCK(ctx, launch_quantile_rank(s.d_sel, H, uint32_t(r_lo), uint32_t(r_hi), d_rank, s.stream));
    HIPCK(ctx, hipMemcpyAsync(s.h_quant, d_thr, sizeof(uint32_t) * 4 * H, hipMemcpyDeviceToHost, s.stream));
    HIPCK(ctx, hipStreamSynchronize(s.stream));
    return FDAS_OK;
  };
  if (s.launched && !s.gated && !s.delivered) {
    if ((st = drain(ctx, s)) != FDAS_OK) return st;
    deliver_early(ctx, s);
  }
  const StampOps times = hsum_stamps(s);
  s.cands_valid = false;  // the lists will belong to these thresholds, not to a search
  std::vector<float> thr(H, -INFINITY);
  fill_hsum(ctx, s, part, thr.data());
  if ((st = put_jobs(ctx, s, times)) != FDAS_OK) return st;
  const uint32_t nb = hmax_blocks(N, nr);
  HIPCK(ctx, launch_hmax(s.fop, N, ctx->cfg.n_templates, rb, nr, H, s.quant, s.stream));
  HIPCK(ctx, launch_quantile_bound(s.quant, nb, uint32_t(std::min<uint64_t>(want, UINT32_MAX)), H, s.d_hsum, s.d_sel,
                                   d_thr, s.stream));
  if ((st = spill_pass()) != FDAS_OK) return st;
  bool all_fit = true;
  for (uint32_t k = 0; k < H; ++k) all_fit = all_fit && h_rank[k] <= ctx->spill;
  if (!all_fit) {
    // A threshold per plane with count(HP_k > t) >= want that fits the spill lists: the
    // planes that overflow are bisected over the bit patterns of non-negative floats,
    // where each pass counts all planes.
    auto value_of = [](int64_t b) { return b < 0 ? -INFINITY : __builtin_bit_cast(float, uint32_t(b)); };
    std::vector<int64_t> lo_b(H), hi_b(H, 0x7f800000);  // count(> lo) >= want, count(> hi) < want
    std::vector<uint32_t> lo_count(h_rank, h_rank + H);
    for (uint32_t k = 0; k < H; ++k) lo_b[k] = h_thr[k] < 0.f ? -1 : int64_t(__builtin_bit_cast(uint32_t, h_thr[k]));
    for (;;) {
      bool fit = true;
      std::vector<int64_t> at(lo_b);
      for (uint32_t k = 0; k < H; ++k) {
        if (lo_count[k] > ctx->spill) {
          fit = false;
          if (hi_b[k] - lo_b[k] <= 1)
            return fail(ctx, FDAS_EOVERFLOW, "plane %u: %u values tie at the quantile, beyond the spill capacity %u",
                        k + 1, lo_count[k], ctx->spill);
          at[k] = lo_b[k] + (hi_b[k] - lo_b[k]) / 2;
        }
        thr[k] = value_of(at[k]);
      }
      // the last pass spills at the final thresholds
      fill_hsum(ctx, s, part, thr.data());
      if ((st = put_jobs(ctx, s)) != FDAS_OK) return st;
      if ((st = spill_pass()) != FDAS_OK) return st;
      if (fit) break;
      for (uint32_t k = 0; k < H; ++k) {
        if (at[k] == lo_b[k]) continue;
        if (h_rank[k] >= want) {
          lo_b[k] = at[k];
          lo_count[k] = h_rank[k];
        } else {
          hi_b[k] = at[k];
        }
      }
    }
  }
  for (uint32_t k = 0; k < H; ++k) {
    const uint32_t c = h_rank[k];
    if (c > ctx->spill)
      return fail(ctx, FDAS_EOVERFLOW, "plane %u: %u values above the bound exceed the spill capacity %u", k + 1, c,
                  ctx->spill);
    if (r_lo >= c) return fail(ctx, FDAS_EDEVICE, "plane %u: only %u values spilled, need %llu", k + 1, c,
                               (unsigned long long)(r_lo + 1));
    const double lo = __builtin_bit_cast(float, h_rank[H + k]), hi = __builtin_bit_cast(float, h_rank[2 * H + k]);
    thresholds[k] = float(lo * (1.0 - g) + hi * g);
  }
  return FDAS_OK;
}

extern "C" fdas_status fdas_get_stage_times(fdas_ctx* ctx, int set, float* ms6) {
  CHECK_SET(ctx, set);
  if (!ms6) return fail(ctx, FDAS_EINVAL, "null output");
  const DevSet& s = ctx->set[set];
  ms6[0] = elapsed(ctx, s, ST_START, ST_INPUT);
  ms6[1] = elapsed(ctx, s, ST_FTC_K, ST_FTC);
  ms6[2] = elapsed(ctx, s, ST_HSUM_K0, ST_HSUM_K1);
  ms6[3] = elapsed(ctx, s, ST_HSUM_K1, ST_ENDS);
  ms6[4] = 0.f;  // the selection writes the lists to host memory
  ms6[5] = elapsed(ctx, s, ST_START, ST_ENDS);
  return FDAS_OK;
}

extern "C" void fdas_print_stats(fdas_ctx* ctx, int set, int reset) {
  if (!ctx || (set != FDAS_SET_A && set != FDAS_SET_B)) return;
  const DevSet& s = ctx->set[set];
  const float t0 = since_epoch(ctx, s, ST_START), t1 = since_epoch(ctx, s, ST_ENDS);
  if (reset) {
    ctx->pipeline_start = t0;
    ctx->pipeline_accum = 0.f;
    ctx->pipeline_launches = 1;
  } else {
    ++ctx->pipeline_launches;
  }
  const float acc = t1 - ctx->pipeline_start;
  info(ctx, "Launch  #%u%c complete @ %.3f ms II ~ %.3f ms", ctx->pipeline_launches, set == FDAS_SET_A ? 'A' : 'B',
       double(acc), double(acc - ctx->pipeline_accum));
  info(ctx, "  Preparation duration: %.3f ms", double(elapsed(ctx, s, ST_START, ST_INPUT)));
  info(ctx, "  FT convolution and IFFT duration: %.3f ms", double(elapsed(ctx, s, ST_FTC_K, ST_FTC)));
  info(ctx, "  Harmonic summing duration: %.3f ms", double(elapsed(ctx, s, ST_HSUM_K0, ST_ENDS)));
  info(ctx, "  Total duration: %.3f ms", double(elapsed(ctx, s, ST_START, ST_ENDS)));
  ctx->pipeline_accum = acc;
}

extern "C" void fdas_print_events(fdas_ctx* ctx, int set) {
  if (!ctx || !ctx->log || (set != FDAS_SET_A && set != FDAS_SET_B)) return;
  const DevSet& s = ctx->set[set];
  float t[ST_ENDS + 1];
  for (int i = 0; i <= ST_ENDS; ++i) t[i] = since_epoch(ctx, s, i);
  char buf[256];
  std::snprintf(buf, sizeof(buf), "@@@,%c,%.6f,%.6f,%.6f,%.6f,%.6f,%.6f,%.6f,%.6f", set == FDAS_SET_A ? 'A' : 'B',
                double(t[ST_START]), double(t[ST_INPUT]), double(t[ST_FTC_K]), double(t[ST_FTC]),
                double(t[ST_HSUM_K0]), double(t[ST_HSUM_K1]), double(t[ST_ENDS]), double(t[ST_ENDS]));
  emit(ctx, FDAS_LOG_INFO, buf);
}

extern "C" int fdas_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

extern "C" fdas_status fdas_device_info(int device, char* name, size_t len, char* arch, size_t arch_len) {
  const int n = fdas_device_count();
  if (device < 0 || device >= n) return FDAS_EINVAL;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
    (void)hipGetLastError();
    return FDAS_EDEVICE;
  }
  if (name && len) {
    std::snprintf(name, len, "%s", prop.name[0] ? prop.name : prop.gcnArchName);
  }
  if (arch && arch_len) std::snprintf(arch, arch_len, "%s", prop.gcnArchName);
  return FDAS_OK;
}

extern "C" const char* fdas_platform_version(void) {
  static char buf[64] = {0};
  if (!buf[0]) {
    int v = 0;
    if (hipRuntimeGetVersion(&v) != hipSuccess) (void)hipGetLastError();
    std::snprintf(buf, sizeof(buf), "HIP %d.%d.%d", v / 10000000, (v / 100000) % 100, v % 100000);
  }
  return buf;
}
