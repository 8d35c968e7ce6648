// Device front end: dedispersed time series -> the spectrum the search takes,
// X[f] = DFT_Ns(s)[f] / Ns for f < N, Ns = 2N (ft_conv.py:123-146), in FP32 on
// the GPU (the reference computes it in FP32 too: scipy.fft.fft of float32
// samples returns complex64).
//
// The 2N real samples are read as N complex points z[n] = s[2n] + i s[2n+1]
// (the float32 array reinterpreted, no copy).  Z = DFT_N(z) uses the four-step
// factorisation N = N1 * N2, and X follows from Z[f] and Z[N-f]:
// X[f] = (E[f] + W_Ns^f O[f]) / Ns with E = (Z[f] + conj Z[N-f]) / 2 and
// O = (Z[f] - conj Z[N-f]) / (2i), the even/odd-sample split of a real DFT.
//   cols_kernel  DFT_N1 down the columns n2 of z [N1][N2], x W_N^(n2 k1)
//   rows_kernel  DFT_N2 along the rows k1, the split, stored in natural order
// N <= 4096 is one row (N1 = 1), N < 16 goes through a radix-2 kernel.
//
// Bound by memory passes: a workgroup of cols_kernel takes kCols neighbouring
// columns and one of rows_kernel a few neighbouring rows together with the rows
// that mirror them, so both transposes and the split happen in the two passes
// that the transforms need anyway.  N = 2^22: 41 us of kernels, 3.4 TB/s, against 88
// with separate transposes and split (six passes of 2 x 8N bytes); the call takes 51 us,
// against 95, on buffers that stay in the last-level cache, and 64, against 98, on
// others each time; N = 2^15: 20 us, against 31, on either.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <string>
#include <vector>

#include "fdas_host.h"
#include "fdas_plan.h"
#include "fft_tile.h"

namespace fdas {
namespace {

// e^(-2 pi i m / 2^log2n) for 0 <= m < 2^log2n, 1 <= log2n <= 23.  The turn is
// reduced in integers to a quarter q and a rest r (in half turns, |r| <= 1/4)
// that FP32 holds exactly; sin(pi r) and cos(pi r) are their Taylor series to
// r^9 and r^10, which leave less than 4e-9.  pi enters in two parts, so that both come
// out within about 0.6 ulp.  In place of sincospif it takes a column pass over 2^22
// points from 20.3 to 19.5 us.
__device__ __forceinline__ float2 root_of_unity(uint32_t m, int log2n) {
  const uint32_t turn = m << (32 - log2n);           // 2^32 a full turn
  const uint32_t q = (turn + 0x20000000u) >> 30;     // nearest quarter (mod 4)
  const float r = float(int32_t(turn - (q << 30))) * 0x1p-31f;
  const float r2 = r * r;
  // sin(pi r) = r (pi + r2 S), pi = 3.14159274 - 8.74227766e-8
  float s = fmaf(r2, 0.0821458866f, -0.5992645293f);
  s = fmaf(r2, s, 2.5501640399f);
  s = fmaf(r2, s, -5.1677127800f);
  s = fmaf(r2, s, -8.74227766e-8f);
  s = fmaf(r, 3.14159274f, r * s);
  float c = fmaf(r2, -0.0258068914f, 0.2353306304f);
  c = fmaf(r2, c, -1.3352627689f);
  c = fmaf(r2, c, 4.0587121264f);
  c = fmaf(r2, c, -4.9348022005f);
  c = fmaf(r2, c, 1.0f);
  // angle q quarters + r: (cos, sin) is (c, s), (-s, c), (-c, -s), (s, -c)
  const bool odd = (q & 1u) != 0;
  const float re = odd ? s : c, im = odd ? c : s;
  const uint32_t re_sign = ((q + 1u) << 30) & 0x80000000u, im_sign = (q << 30) & 0x80000000u;
  return make_float2(__uint_as_float(__float_as_uint(re) ^ re_sign),
                     __uint_as_float(__float_as_uint(im) ^ im_sign ^ 0x80000000u));
}

// DFT-R of v[O .. O + R-1], natural order.
template <int R, int O>
__device__ __forceinline__ void dft_group(float2 (&v)[16]) {
  if constexpr (R == 2) {
    const float2 a = v[O], b = v[O + 1];
    v[O] = cadd(a, b);
    v[O + 1] = csub(a, b);
  } else {
    dftD<-1, R, O>(v);
  }
}
template <int R, int O = 0>
__device__ __forceinline__ void dft_groups(float2 (&v)[16]) {
  if constexpr (R > 1) {
    dft_group<R, O>(v);
    if constexpr (O + R < 16) dft_groups<R, O + R>(v);
  }
}

// Forward DFT of G lines of L = 16 NT points by a workgroup of NT * G threads:
// thread (b, g) holds 16 points of line g.  Two register passes (DFT-16, DFT-NT)
// up to L = 256, three (DFT-16, DFT-16, DFT-D) beyond, with LDS exchanges whose
// lines are interleaved ([point][g]): consecutive lanes hold neighbouring lines,
// as they do in memory, and touch consecutive banks.
template <int L, int G>
struct LineFFT {
  static constexpr int NT = L / 16;
  static constexpr bool THREE = NT > 16;
  static constexpr int D = THREE ? NT / 16 : NT;  // radix of the last pass
  static constexpr int RS = NT + 1;               // row stride of the [ka][b] exchange
  static constexpr int LDS_ELEMS = 16 * RS * G;   // >= L * G

  // Frequency bin of register slot `slot` of thread b.
  __device__ static constexpr int slot_bin(int b, int slot) {
    return b + NT * (slot / D) + (THREE ? 256 : 16) * (slot % D);
  }

  // v[a] = line g's point NT * a + b.  Ends with a barrier after the last LDS read.
  __device__ __forceinline__ static void forward(float2 (&v)[16], float2* __restrict__ lds, int b, int g,
                                                 const float2* __restrict__ tw1, const float2* __restrict__ tw2) {
    dft16<-1>(v);
    if constexpr (NT > 1) {
#pragma unroll
      for (int k = 1; k < 16; ++k) v[k] = cmul(v[k], gld2(tw1, size_t(k * NT + b)));
#pragma unroll
      for (int k = 0; k < 16; ++k) lds[(k * RS + b) * G + g] = v[k];
      __syncthreads();
      if constexpr (THREE) {
        const int ka = b & 15, d = b >> 4;
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = lds[(ka * RS + D * c + d) * G + g];
        __syncthreads();
        dft16<-1>(v);
#pragma unroll
        for (int k = 1; k < 16; ++k) v[k] = cmul(v[k], gld2(tw2, size_t(k * D + d)));
#pragma unroll
        for (int kc = 0; kc < 16; ++kc) lds[(d * 256 + 16 * kc + ka) * G + g] = v[kc];
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 16; ++s) v[s] = lds[((s % D) * 256 + b + NT * (s / D)) * G + g];
      } else {
#pragma unroll
        for (int s = 0; s < 16; ++s) v[s] = lds[((b + NT * (s / D)) * RS + s % D) * G + g];
      }
      __syncthreads();
      dft_groups<D>(v);
    }
  }
};

// Workgroups in units of 4 neighbours per die: their lines share 128-byte cache
// lines (kCols * 8 bytes each), which meet in one die's L2 this way.
__device__ __forceinline__ uint32_t die_units(uint32_t blk, uint32_t n) {
  const uint32_t i = blk >> 3;
  return n % 32u == 0 ? (i >> 2) * 32u + (blk & 7u) * 4u + (i & 3u) : blk;
}

// Columns of one cols_kernel workgroup and rows of one rows_kernel workgroup (half of
// them mirrors).  At N = 2^22, on buffers that stay in the last-level cache, the call took
// 52 us with 4 and 8, 52 with 8 and 8, 56 with 4 and 4, 55 with 8 and 4; at 2^20 31, 33, 31, 32.
constexpr int kCols = 4;
constexpr int kRows = 8;

// z [L][n2] -> A, column n2 transformed and times W_N^(n2 k1), N = 2^log2n = L n2.
// A is laid out [n2 / kCols][k1][n2 % kCols]: whole lines are stored, and a group
// of neighbouring rows k1 is read back in runs of kCols times their number.
template <int L>
__global__ __launch_bounds__(L / 16 * kCols) void cols_kernel(const float2* __restrict__ z, float2* __restrict__ A,
                                                              uint32_t n2, int log2n,
                                                              const float2* __restrict__ tw1,
                                                              const float2* __restrict__ tw2) {
  using F = LineFFT<L, kCols>;
  __shared__ float2 lds[F::LDS_ELEMS];
  const int g = int(threadIdx.x) % kCols, b = int(threadIdx.x) / kCols;
  const uint32_t w = die_units(blockIdx.x, gridDim.x);
  const uint32_t col = w * kCols + uint32_t(g);
  float2 v[16];
#pragma unroll
  for (int a = 0; a < 16; ++a) v[a] = gld2(z, size_t(F::NT * a + b) * n2 + col);
  F::forward(v, lds, b, g, tw1, tw2);
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const uint32_t k1 = uint32_t(F::slot_bin(b, s));
    const float2 y = cmul(v[s], root_of_unity(col * k1, log2n));  // col * k1 < N
    ((FDAS_GLOBAL fdas_vf2*)A)[(size_t(w) * L + k1) * kCols + uint32_t(g)] = fdas_vf2{y.x, y.y};
  }
}

// Rows k1 of A, R per workgroup: transformed, split and stored.  The workgroup
// takes rows j .. j + R/2 - 1 and their mirrors n1 - j - R/2 + 1 .. n1 - j, since
// Z[N - f] of f = k1 + n1 k2 is row n1 - k1, bin L-1 - k2; the first one, whose row
// 0 mirrors itself, has row n1 / 2, the other such row, in the place of row n1.
// Each thread forms both X[f] and X[N - f] for its bins k2 < L/2, from
// X[f] = E + T and X[N - f] = conj(E - T), T = W_Ns^f O.  R = 1: n1 = 1, A = z.
template <int L, int R>
__global__ __launch_bounds__(L / 16 * R) void rows_kernel(const float2* __restrict__ A, float2* __restrict__ X,
                                                          uint32_t n1, int log2n, float inv_ns,
                                                          const float2* __restrict__ tw1,
                                                          const float2* __restrict__ tw2) {
  using F = LineFFT<L, R>;
  __shared__ float2 lds[F::LDS_ELEMS];
  const int g = int(threadIdx.x) % R, b = int(threadIdx.x) / R;
  uint32_t row = 0;
  int mirror = 0;
  float2 v[16];
  if constexpr (R == 1) {
#pragma unroll
    for (int a = 0; a < 16; ++a) v[a] = gld2(A, size_t(F::NT * a + b));
  } else {
    const uint32_t j = die_units(blockIdx.x, gridDim.x) * uint32_t(R / 2);
    row = g < R / 2 ? j + uint32_t(g) : n1 - j - uint32_t(R - 1 - g);
    mirror = R - 1 - g;
    if (row == n1) row = n1 / 2;
    if (row == 0 || row == n1 / 2) mirror = g;
#pragma unroll
    for (int a = 0; a < 16; ++a) {
      const uint32_t col = uint32_t(F::NT * a + b);
      v[a] = gld2(A, (size_t(col / kCols) * n1 + row) * kCols + col % kCols);
    }
  }
  F::forward(v, lds, b, g, tw1, tw2);
#pragma unroll
  for (int s = 0; s < 16; ++s) lds[F::slot_bin(b, s) * R + g] = v[s];
  __syncthreads();
  const uint32_t n = 1u << log2n;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    if (F::slot_bin(0, s) >= L / 2) continue;  // k2 >= L/2: its mirror's thread forms both
    const uint32_t k2 = uint32_t(F::slot_bin(b, s)), f = row + n1 * k2;
    const uint32_t m2 = row == 0 ? (L - k2) & (L - 1u) : L - 1u - k2;
    const float2 p = v[s], q = lds[m2 * R + uint32_t(mirror)];
    const float2 e = make_float2(0.5f * (p.x + q.x), 0.5f * (p.y - q.y));
    const float2 o = make_float2(0.5f * (p.y + q.y), -0.5f * (p.x - q.x));
    const float2 t = cmul(root_of_unity(f, log2n + 1), o);  // W_Ns^f, Ns = 2N
    const float2 x = cadd(e, t), y = csub(e, t);
    ((FDAS_GLOBAL fdas_vf2*)X)[f] = fdas_vf2{x.x * inv_ns, x.y * inv_ns};
    if (f != 0) {
      ((FDAS_GLOBAL fdas_vf2*)X)[n - f] = fdas_vf2{y.x * inv_ns, -y.y * inv_ns};
    } else {  // X[N] is not stored; bin N/2 mirrors itself, W_Ns^(N/2) = -i
      const float2 h = lds[(L / 2) * R + g];
      ((FDAS_GLOBAL fdas_vf2*)X)[n / 2] = fdas_vf2{h.x * inv_ns, -h.y * inv_ns};
    }
  }
}

constexpr int kLdsFftMax = 8;
constexpr int kLdsFftThreads = 64;

__device__ __forceinline__ uint32_t bit_reverse(uint32_t i, int bits) { return __brev(i) >> (32 - bits); }

// One L-point forward DFT, L = 2^log2l <= 8, radix-2 in LDS.
__global__ __launch_bounds__(kLdsFftThreads) void ldsfft_kernel(const float2* __restrict__ in, float2* __restrict__ out,
                                                                int log2l) {
  __shared__ float2 buf[kLdsFftMax];
  const uint32_t L = 1u << log2l, tid = threadIdx.x;
  if (tid < L) buf[log2l ? bit_reverse(tid, log2l) : 0] = gld2(in, tid);
  __syncthreads();
  for (int s = 1; s <= log2l; ++s) {
    const uint32_t half = 1u << (s - 1);
    if (tid < L / 2) {
      const uint32_t pos = tid & (half - 1u);
      const uint32_t i0 = ((tid >> (s - 1)) << s) + pos, i1 = i0 + half;
      const float2 t = cmul(root_of_unity(pos, s), buf[i1]);
      const float2 u = buf[i0];
      buf[i0] = cadd(u, t);
      buf[i1] = csub(u, t);
    }
    __syncthreads();
  }
  if (tid < L) ((FDAS_GLOBAL fdas_vf2*)out)[tid] = fdas_vf2{buf[tid].x, buf[tid].y};
}

// X[f] = (E + W_Ns^f O) / Ns from the N-point transform Z of the packed series.
__global__ __launch_bounds__(256) void real_spectrum_kernel(const float2* __restrict__ Z, float2* __restrict__ X,
                                                            uint32_t n, int log2n, float inv_ns) {
  for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < n; f += gridDim.x * blockDim.x) {
    const float2 a = gld2(Z, f);
    const float2 b = gld2(Z, (n - f) & (n - 1u));  // Z[N - f], Z[N] = Z[0]
    // E = (a + conj b) / 2, O = (a - conj b) / (2i)
    const float2 e = make_float2(0.5f * (a.x + b.x), 0.5f * (a.y - b.y));
    const float2 o = make_float2(0.5f * (a.y + b.y), -0.5f * (a.x - b.x));
    const float2 w = root_of_unity(f, log2n + 1);  // W_Ns^f, Ns = 2N
    const float2 x = cadd(e, cmul(w, o));
    ((FDAS_GLOBAL fdas_vf2*)X)[f] = fdas_vf2{x.x * inv_ns, x.y * inv_ns};
  }
}

int ilog2(uint32_t v) {
  int l = 0;
  while ((1u << l) < v) ++l;
  return l;
}

}  // namespace
}  // namespace fdas

using namespace fdas;

struct fdas_frontend {
  uint32_t n = 0, n1 = 0, n2 = 0;
  int device = 0;
  std::string last_error;
  hipStream_t stream = nullptr;
  LineTables tables;           // kept until the copy to the device has surely been made
  float2* mem = nullptr;       // the tables, then buf
  float2* buf = nullptr;       // N points between the two passes
  float2* series = nullptr;    // device copy of a host series
  float2* spectrum = nullptr;  // device result for a host destination
  const float2* tw1[2] = {nullptr, nullptr};  // twiddles of the column (n1) and row (n2) transforms
  const float2* tw2[2] = {nullptr, nullptr};
};

namespace {

fdas_status fe_fail(fdas_frontend* fe, fdas_status st, const char* fmt, ...) {
  char b[512];
  va_list ap;
  va_start(ap, fmt);
  std::vsnprintf(b, sizeof(b), fmt, ap);
  va_end(ap);
  if (fe) fe->last_error = std::string("[ERROR] ") + b;
  return st;
}

#define FEHIP(fe, expr)                                                                                          \
  do {                                                                                                           \
    hipError_t e_ = (expr);                                                                                      \
    if (e_ != hipSuccess)                                                                                        \
      return fe_fail(fe, FDAS_EDEVICE, "HIP call failed with status %d (%s): %s", int(e_), hipGetErrorString(e_), \
                     #expr);                                                                                     \
  } while (0)

template <int L>
void launch_cols(const fdas_frontend* fe, const float2* z, int log2n) {
  hipLaunchKernelGGL(cols_kernel<L>, dim3(fe->n2 / kCols), dim3(L / 16 * kCols), 0, fe->stream, z, fe->buf, fe->n2,
                     log2n, fe->tw1[0], fe->tw2[0]);
}

template <int L, int R>
void launch_rows(const fdas_frontend* fe, const float2* in, float2* X, int log2n) {
  hipLaunchKernelGGL((rows_kernel<L, R>), dim3(R == 1 ? 1 : fe->n1 / R), dim3(L / 16 * R), 0, fe->stream, in, X, fe->n1,
                     log2n, 1.0f / float(2.0 * fe->n), fe->tw1[1], fe->tw2[1]);
}

// X from z (N >= 16).
fdas_status transform(fdas_frontend* fe, const float2* z, float2* X, int log2n) {
  if (fe->n1 == 1) {
    switch (fe->n2) {
      case 16: launch_rows<16, 1>(fe, z, X, log2n); break;
      case 32: launch_rows<32, 1>(fe, z, X, log2n); break;
      case 64: launch_rows<64, 1>(fe, z, X, log2n); break;
      case 128: launch_rows<128, 1>(fe, z, X, log2n); break;
      case 256: launch_rows<256, 1>(fe, z, X, log2n); break;
      case 512: launch_rows<512, 1>(fe, z, X, log2n); break;
      case 1024: launch_rows<1024, 1>(fe, z, X, log2n); break;
      case 2048: launch_rows<2048, 1>(fe, z, X, log2n); break;
      case 4096: launch_rows<4096, 1>(fe, z, X, log2n); break;
      default: return fe_fail(fe, FDAS_EINVAL, "no transform of %u points", fe->n2);
    }
    FEHIP(fe, hipGetLastError());
    return FDAS_OK;
  }
  switch (fe->n1) {
    case 64: launch_cols<64>(fe, z, log2n); break;
    case 128: launch_cols<128>(fe, z, log2n); break;
    case 256: launch_cols<256>(fe, z, log2n); break;
    case 512: launch_cols<512>(fe, z, log2n); break;
    case 1024: launch_cols<1024>(fe, z, log2n); break;
    case 2048: launch_cols<2048>(fe, z, log2n); break;
    default: return fe_fail(fe, FDAS_EINVAL, "no column transform of %u points", fe->n1);
  }
  FEHIP(fe, hipGetLastError());
  switch (fe->n2) {
    case 128: launch_rows<128, kRows>(fe, fe->buf, X, log2n); break;
    case 256: launch_rows<256, kRows>(fe, fe->buf, X, log2n); break;
    case 512: launch_rows<512, kRows>(fe, fe->buf, X, log2n); break;
    case 1024: launch_rows<1024, kRows>(fe, fe->buf, X, log2n); break;
    case 2048: launch_rows<2048, kRows>(fe, fe->buf, X, log2n); break;
    default: return fe_fail(fe, FDAS_EINVAL, "no row transform of %u points", fe->n2);
  }
  FEHIP(fe, hipGetLastError());
  return FDAS_OK;
}

fdas_status fe_init(fdas_frontend* fe) {
  FEHIP(fe, hipSetDevice(fe->device));
  FEHIP(fe, hipStreamCreateWithFlags(&fe->stream, hipStreamNonBlocking));
  // One allocation and one copy, enqueued before anything that reads it.  Creation takes 23 / 27 / 41 / 69 us at 2^7 /
  // 2^15 / 2^18 / 2^22 bins; with an allocation and a blocking copy per table, some made twice or never read, it took
  // 34 / 65 / 101 / 144.
  fe->tables = line_tables({fe->n1, fe->n2});
  const std::vector<float2>& t = fe->tables.data;
  const size_t table_elems = (t.size() + 31) / 32 * 32;  // buf on a 256-byte boundary
  FEHIP(fe, hipMalloc(&fe->mem, sizeof(float2) * (table_elems + fe->n)));
  fe->buf = fe->mem + table_elems;
  if (!t.empty())
    FEHIP(fe, hipMemcpyAsync(fe->mem, t.data(), sizeof(float2) * t.size(), hipMemcpyHostToDevice, fe->stream));
  for (int i = 0; i < 2; ++i) {
    fe->tw1[i] = fe->mem + fe->tables.w1[i];
    fe->tw2[i] = fe->mem + fe->tables.w2[i];
  }
  return FDAS_OK;
}

}  // namespace

extern "C" {

fdas_status fdas_frontend_create(uint32_t n_bins, int device, fdas_frontend** out) {
  if (!out) return FDAS_EINVAL;
  *out = nullptr;
  if (n_bins < 2 || n_bins > (1u << 22) || (n_bins & (n_bins - 1u))) return FDAS_EINVAL;
  int n_dev = 0;
  if (hipGetDeviceCount(&n_dev) != hipSuccess || device < 0 || device >= n_dev) {
    (void)hipGetLastError();
    return FDAS_EDEVICE;
  }
  auto* fe = new fdas_frontend();
  fe->n = n_bins;
  fe->device = device;
  // One workgroup up to 4096 points, then lengths as equal as they can be (64 x 128 .. 2048 x 2048).
  fe->n1 = n_bins <= 4096 ? 1u : 1u << (ilog2(n_bins) / 2);
  fe->n2 = n_bins / fe->n1;
  if (fe_init(fe) != FDAS_OK) {
    fdas_frontend_destroy(fe);
    return FDAS_EDEVICE;
  }
  *out = fe;
  return FDAS_OK;
}

void fdas_frontend_destroy(fdas_frontend* fe) {
  if (!fe) return;
  (void)hipSetDevice(fe->device);
  if (fe->stream) (void)hipStreamSynchronize(fe->stream);
  for (float2* p : {fe->mem, fe->series, fe->spectrum}) (void)hipFree(p);
  if (fe->stream) (void)hipStreamDestroy(fe->stream);
  delete fe;
}

const char* fdas_frontend_last_error(const fdas_frontend* fe) { return fe ? fe->last_error.c_str() : "null front end"; }

fdas_status fdas_frontend_run(fdas_frontend* fe, const float* series, uint32_t flags, void* spectrum_c64) {
  if (!fe) return FDAS_EINVAL;
  if (!series || !spectrum_c64) return fe_fail(fe, FDAS_EINVAL, "null series or spectrum");
  FEHIP(fe, hipSetDevice(fe->device));
  const uint32_t N = fe->n;
  const int log2n = ilog2(N);
  const float2* z = reinterpret_cast<const float2*>(series);
  if (!(flags & FDAS_FE_DEVICE_INPUT)) {
    if (!fe->series) FEHIP(fe, hipMalloc(&fe->series, sizeof(float2) * N));
    FEHIP(fe, hipMemcpyAsync(fe->series, series, sizeof(float2) * N, hipMemcpyHostToDevice, fe->stream));
    z = fe->series;
  }
  float2* X = static_cast<float2*>(spectrum_c64);
  if (!(flags & FDAS_FE_DEVICE_OUTPUT)) {
    if (!fe->spectrum) FEHIP(fe, hipMalloc(&fe->spectrum, sizeof(float2) * N));
    X = fe->spectrum;
  }
  if (N >= 16) {
    const fdas_status st = transform(fe, z, X, log2n);
    if (st != FDAS_OK) return st;
  } else {
    hipLaunchKernelGGL(ldsfft_kernel, dim3(1), dim3(kLdsFftThreads), 0, fe->stream, z, fe->buf, log2n);
    FEHIP(fe, hipGetLastError());
    hipLaunchKernelGGL(real_spectrum_kernel, dim3(1), dim3(kLdsFftThreads), 0, fe->stream, fe->buf, X, N, log2n,
                       1.0f / float(2.0 * N));
    FEHIP(fe, hipGetLastError());
  }
  if (!(flags & FDAS_FE_DEVICE_OUTPUT))
    FEHIP(fe, hipMemcpyAsync(spectrum_c64, X, sizeof(float2) * N, hipMemcpyDeviceToHost, fe->stream));
  FEHIP(fe, hipStreamSynchronize(fe->stream));
  return FDAS_OK;
}

}  // extern "C"
