// Host-side test of the engine's own code under sanitizers, with a HIP runtime of host memory in which every kernel
// launch only reads its job descriptors (and the selection writes one entry per list): autotuning, an eager plan
// twice, a changed request, served requests, and plans launched while requests are served.  An event counts as
// reached 1 ms after its record, so that work is in flight for a while: kernels of plans (launched by the main thread)
// and of served groups (by the scheduler's) must not be in flight together.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "fdas.h"
#include "fdas_kernels.h"

static int failures = 0;
#define CHECK(cond)                                                                   \
  do {                                                                                \
    if (!(cond)) ++failures, std::printf("FAIL line %d: %s\n", __LINE__, #cond);      \
  } while (0)

typedef std::chrono::steady_clock Clock;
static const std::thread::id main_thread = std::this_thread::get_id();
static int kind() { return std::this_thread::get_id() == main_thread ? 0 : 1; }
static std::mutex mu;
static int n_launched[2] = {0, 0}, n_reached[2] = {0, 0};  // kernels launched; known to have ended
struct Event {
  int kind = 0, launched = 0;
  Clock::time_point at{};
};
static void launched() {
  std::lock_guard<std::mutex> lk(mu);
  const int k = kind();
  CHECK(n_reached[1 - k] == n_launched[1 - k]);  // nothing of the other kind is in flight
  ++n_launched[k];
}
static void reached(const Event& e) {
  std::lock_guard<std::mutex> lk(mu);
  if (e.launched > n_reached[e.kind]) n_reached[e.kind] = e.launched;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return *p = std::malloc(n), *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) { return std::memset(p, 0, sizeof(*p)), hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(new Event), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<Event*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  *reinterpret_cast<Event*>(e) = {kind(), n_launched[kind()], Clock::now() + std::chrono::milliseconds(1)};
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  if (Clock::now() < reinterpret_cast<Event*>(e)->at) return hipErrorNotReady;
  return reached(*reinterpret_cast<Event*>(e)), hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::this_thread::sleep_until(reinterpret_cast<Event*>(e)->at);
  return reached(*reinterpret_cast<Event*>(e)), hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(std::malloc(1)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
}

namespace fdas {
hipError_t launch_ftconv(int, const FtcJob* j, uint32_t n, uint32_t items, const float2*, const float2*, uint32_t,
                         hipStream_t, uint64_t*) {
  launched();
  CHECK(n > 0 && j[n - 1].item_begin + j[n - 1].n_tiles * j[n - 1].n_chunks == items);
  for (uint32_t i = 0; i < n; ++i) CHECK(j[i].spectrum && j[i].fop && j[i].hperm);
  return hipSuccess;
}
hipError_t launch_hsum(const HsumJob* j, uint32_t n, uint32_t blocks, uint32_t H, hipStream_t, uint64_t*) {
  launched();
  for (uint32_t i = 0; i < n; ++i) {
    CHECK(j[i].n_harmonics == H && j[i].block_begin < blocks);
    j[i].counts[(H - 1) * kPlaneCounters] = 0;
    j[i].spill_key[size_t(H) * j[i].spill_cap - 1] = 0;
    j[i].spill_pwr[size_t(H) * j[i].spill_cap - 1] = 0.f;
  }
  return hipSuccess;
}
hipError_t launch_select(const SelectJob* j, uint32_t n, uint32_t cap, hipStream_t, uint64_t*, uint64_t*) {
  launched();
  for (uint32_t i = 0; i < n; ++i) {
    CHECK(j[i].cap == cap);
    j[i].hist[kSelectBins - 1] = 0;
    j[i].compact_key[j[i].compact_cap - 1] = 0;
    j[i].compact_pwr[j[i].compact_cap - 1] = 0.f;
    j[i].out_key[0] = i + 1;
    j[i].out_key[cap - 1] = i + 1;
    j[i].out_pwr[0] = j[i].out_pwr[cap - 1] = j[i].thr;
    *j[i].out_n = 1;
    *j[i].out_count = 1;
  }
  return hipSuccess;
}
hipError_t launch_fused(const FtcJob*, uint32_t, uint32_t, const float2*, const float2*, const HsumJob*, uint32_t,
                        uint32_t, uint32_t, hipStream_t) {
  return hipErrorNotSupported;
}
bool fused_supported(uint32_t, uint32_t, bool) { return false; }
hipError_t launch_zero_u32(uint32_t* p, uint32_t n, hipStream_t) { return std::memset(p, 0, 4ull * n), hipSuccess; }
hipError_t launch_clear_counters(const SelectJob* j, uint32_t n, hipStream_t) {
  for (uint32_t i = 0; i < n; ++i) {
    std::memset(j[i].hist, 0, 4ull * kSelectBins);
    *j[i].compact_n = 0;
    *const_cast<uint32_t*>(j[i].count) = 0;
  }
  return hipSuccess;
}
}  // namespace fdas

int main() {
  constexpr uint32_t T = 5, TAPS = 9, N = 3001, CAP = 16;
  std::vector<float> taps(2 * T * TAPS, 1.f), x(2 * N, 1.f);
  for (uint32_t schedule : {FDAS_SCHEDULE_LAGGED, FDAS_SCHEDULE_STREAMS}) {
    fdas_engine_config cfg;
    fdas_engine_default_config(&cfg);
    cfg.cands_per_harmonic = CAP;
    cfg.spill_per_harmonic = 64;
    cfg.group_trials = 2;
    cfg.groups_in_flight = 2;
    cfg.hbm_budget_bytes = 256ull << 20;
    cfg.plan_schedule = schedule;
    fdas_engine* e = nullptr;
    CHECK(fdas_engine_create(&cfg, nullptr, nullptr, &e) == FDAS_OK);
    uint32_t bank = 0;
    CHECK(fdas_engine_add_bank(e, taps.data(), T, TAPS, &bank) == FDAS_OK);
    CHECK(fdas_engine_prepare(e, N, bank, FDAS_ALL, nullptr) == FDAS_OK);  // autotuned
    constexpr uint32_t R = 5;
    fdas_request req[R] = {};
    fdas_result res[R] = {};
    std::vector<std::vector<uint32_t>> key(R);
    std::vector<std::vector<float>> power(R);
    for (uint32_t i = 0; i < R; ++i) {
      const uint32_t H = i % 2 ? 3 : 16;
      req[i].spectrum = x.data();
      req[i].n_bins = N - 700 * (i / 2);
      req[i].bank = bank;
      req[i].n_harmonics = H;
      req[i].part = FDAS_ALL;
      req[i].tag = i;
      for (uint32_t k = 0; k < H; ++k) req[i].thresholds[k] = float(i + 1);
      key[i].assign(H * CAP, 9);
      power[i].assign(H * CAP, 9.f);
      res[i].key = key[i].data();
      res[i].power = power[i].data();
    }
    auto complete = [&](const fdas_result& r) {
      const uint32_t i = uint32_t(r.tag);
      CHECK(r.status == FDAS_OK && r.n_harmonics == req[i].n_harmonics);
      for (uint32_t p = 0; p < req[i].n_harmonics; ++p) {
        CHECK(r.n_kept[p] == 1 && r.key[p * CAP] != 0 && r.power[p * CAP] == req[i].thresholds[p]);
        for (uint32_t c = 1; c < CAP; ++c) CHECK(r.key[p * CAP + c] == 0 && r.power[p * CAP + c] == 0.f);
      }
    };
    fdas_plan* plan = nullptr;
    CHECK(fdas_plan_create(e, req, R, 0, &plan) == FDAS_OK);
    for (int run = 0; plan && run < 2; ++run) {
      CHECK(fdas_plan_launch(plan) == FDAS_OK && fdas_plan_wait(plan, res) == FDAS_OK);
      for (const fdas_result& r : res) complete(r);
      req[3].thresholds[0] = 77.f;
      CHECK(fdas_plan_set_request(plan, 3, nullptr, req[3].thresholds) == FDAS_OK);
    }
    // requests served while plans run: submitted before, between and after their launches
    fdas_result planned[R];
    std::vector<std::vector<uint32_t>> pkey(key);
    std::vector<std::vector<float>> ppower(power);
    for (uint32_t i = 0; i < R; ++i) {
      planned[i] = res[i];
      planned[i].key = pkey[i].data();
      planned[i].power = ppower[i].data();
    }
    fdas_plan* second = nullptr;
    CHECK(fdas_plan_create(e, req, R, 0, &second) == FDAS_OK);
    for (int round = 0; round < 4; ++round) {
      for (uint32_t i = 0; i < R; ++i) {
        CHECK(fdas_engine_submit(e, &req[i], &res[i]) == FDAS_OK);
        if (i == 1) CHECK(fdas_plan_launch(plan) == FDAS_OK);
        if (i == 3) CHECK(fdas_plan_launch(second) == FDAS_OK);
        if (round % 2) std::this_thread::sleep_for(std::chrono::microseconds(300));
      }
      for (fdas_plan* p : {plan, second}) {
        CHECK(fdas_plan_wait(p, planned) == FDAS_OK);
        for (const fdas_result& r : planned) complete(r);
      }
      for (uint32_t got = 0; got < R;) {
        fdas_result* done[R];
        uint32_t n = 0;
        CHECK(fdas_engine_poll(e, done, R, &n, 1000) == FDAS_OK && n > 0);
        if (n == 0) break;
        for (uint32_t i = 0; i < n; ++i) complete(*done[i]);
        got += n;
      }
    }
    fdas_plan_destroy(plan);
    fdas_plan_destroy(second);
    fdas_engine_destroy(e);
  }
  if (failures == 0) std::printf("engine host test ok\n");
  return failures != 0;
}
