// Intensity-moment reductions, pupils and small utility kernels.
// Moments follow measures.py:1-38 (sums of |u|^2 times a coordinate weight,
// times delta^2) and simulations/beam.py:26-33 (mean_x2_r); pupils follow
// pupils.py:8-13 with the mask (x - sx)^2 + (y + sy)^2 <= a^2.
#include <mutex>

#include "pa_fft.h"
#include "pa_internal.h"

namespace pa {

// Adds the block's NT per-thread values of sums k < K (s_part[k][thread], NT a
// multiple of 64) in a fixed order: 16 threads per sum add NT / 16 values each,
// then the 16 by xor shuffles.  Thread 16 k holds sum k (k < K <= NT / 16).
template <int NT>
__device__ __forceinline__ double block_sums(const double (*s_part)[NT + 1], int K) {
  const int k = threadIdx.x / 16, j = threadIdx.x % 16;
  double a = 0.0;
  if (k < K) {
#pragma unroll
    for (int i = 0; i < NT / 16; ++i) a += s_part[k][j + 16 * i];
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
  return a;
}

// Per-tile partial sums over row-major fields (same format as k_row_last).
// The 8 bytes per element bound it, so the arithmetic per element is kept
// small: a wave walks pieces of 128 columns of one row (one 16-byte load per
// lane, kFPAhead pieces in flight); the moments of a row are sums of I, m I and
// m^2 I with m = c - n/2, folded once per row with the row's y; the pupils are
// the column intervals that circle_cols finds per row (the exact float64
// predicate).  Lane p holds pupil p's interval of the row, so two ballots tell
// which pupils a piece touches and which hold it whole: most pieces touch
// none, and only those that an edge crosses take a test per element.  One
// block per tile, the block's sums added through LDS.
// Measured, four 2048^2 fields with eight pupils: 70 us with every pupil's
// float64 predicate evaluated per element, 26 us (5.2 TB/s) so.
typedef float pa_f4c __attribute__((ext_vector_type(4), aligned(8)));   // two complex64, at 8-byte addresses
constexpr int kFPThreads = 256, kFPAhead = 4;

template <int N, int T>
__global__ void __launch_bounds__(kFPThreads)
k_field_partials(const float2* __restrict__ u, double* __restrict__ part, const double* __restrict__ chparam,
                 const double* __restrict__ pup, int npup, const double* __restrict__ pup_moments,
                 const int* __restrict__ chan) {
  constexpr int NW = kFPThreads / 64, PER = T * N / 2 / kFPThreads;   // pieces per wave
  constexpr int AH = PER < kFPAhead ? PER : kFPAhead;
  constexpr bool SPLIT = N < 128;                                     // a piece spans two rows
  constexpr int RP = SPLIT ? 1 : (PER < N / 128 ? PER : N / 128);     // pieces of one row
  static_assert(PER * NW * 128 == T * N && PER % AH == 0 && PER % RP == 0, "whole pieces and rows");
  __shared__ double s_part[6 + kMaxPupils][kFPThreads + 1];
  __shared__ int2 s_pc[T * kMaxPupils];
  const int b = blockIdx.y, tile = blockIdx.x, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ch = chan ? chan[b] : 0;
  const double delta = chparam[ch * kChParams + 0];
  // piece i of the wave: tile elements e = 128 (wave PER + i) + 2 lane and e + 1
  const pa_f4c* f = reinterpret_cast<const pa_f4c*>(u + (size_t)b * N * N + (size_t)tile * T * N) + wave * PER * 64 + lane;
  pa_f4c nx[AH];
#pragma unroll
  for (int j = 0; j < AH; ++j) nx[j] = f[j * 64];
  if (threadIdx.x < T * kMaxPupils) {
    const int tt = threadIdx.x / kMaxPupils, p = threadIdx.x % kMaxPupils;
    int lo = 0, hi = -1;
    if (p < npup) {
      const double* pp = pup + ((size_t)ch * kMaxPupils + p) * 3;
      const double a = pp[0];
      const double sx = pup_moments ? pup_moments[(size_t)b * kMoments + 1] : pp[1];
      const double sy = pup_moments ? pup_moments[(size_t)b * kMoments + 2] : pp[2];
      circle_cols(N, delta, grid_offset(tile * T + tt, N, delta, -sy), sx, a * a, lo, hi);
    }
    s_pc[threadIdx.x] = make_int2(lo, hi);
  }
  __syncthreads();
  double acc[6], ps[kMaxPupils], r0 = 0.0, r1 = 0.0, r2 = 0.0;   // r: the row's sums of I, m I, m^2 I
#pragma unroll
  for (int k = 0; k < 6; ++k) acc[k] = 0.0;
#pragma unroll
  for (int p = 0; p < kMaxPupils; ++p) ps[p] = 0.0;
  int2 q = make_int2(0, -1);                                      // lane p: the row's interval of pupil p
#pragma unroll 1
  for (int i0 = 0; i0 < PER; i0 += AH) {
    pa_f4c v[AH];
#pragma unroll
    for (int j = 0; j < AH; ++j) v[j] = nx[j];
    if (i0 + AH < PER)
#pragma unroll
      for (int j = 0; j < AH; ++j) nx[j] = f[(i0 + AH + j) * 64];
#pragma unroll
    for (int j = 0; j < AH; ++j) {
      const int e = 128 * (wave * PER + i0 + j), c0 = e % N, c = (e + 2 * lane) % N;
      const int row = SPLIT ? (e + 2 * lane) / N : e / N;
      const double I0 = (double)v[j].x * v[j].x + (double)v[j].y * v[j].y;
      const double I1 = (double)v[j].z * v[j].z + (double)v[j].w * v[j].w;
      const double m0 = (double)(c - N / 2), m1 = m0 + 1.0;
      r0 += I0 + I1;
      r1 += m0 * I0 + m1 * I1;
      r2 += m0 * m0 * I0 + m1 * m1 * I1;
      if constexpr (SPLIT) {
#pragma unroll
        for (int p = 0; p < kMaxPupils; ++p) {
          const int2 w = s_pc[row * kMaxPupils + p];
          ps[p] += (c >= w.x && c <= w.y ? I0 : 0.0) + (c + 1 >= w.x && c + 1 <= w.y ? I1 : 0.0);
        }
      } else {
        if ((i0 + j) % RP == 0 && lane < kMaxPupils) q = s_pc[row * kMaxPupils + lane];
        const unsigned touched = (unsigned)__ballot(q.x < c0 + 128 && q.y >= c0 && q.x <= q.y);
        if (touched) {
          const unsigned whole = (unsigned)__ballot(q.x <= c0 && q.y >= c0 + 127);
#pragma unroll
          for (int p = 0; p < kMaxPupils; ++p) {
            if (whole >> p & 1) {
              ps[p] += I0 + I1;
            } else if (touched >> p & 1) {
              const int lo = __builtin_amdgcn_readlane(q.x, p), hi = __builtin_amdgcn_readlane(q.y, p);
              ps[p] += (c >= lo && c <= hi ? I0 : 0.0) + (c + 1 >= lo && c + 1 <= hi ? I1 : 0.0);
            }
          }
        }
      }
      if ((i0 + j) % RP == RP - 1) {
        const double y = (double)(tile * T + row - N / 2) * delta, x1 = r1 * delta;
        acc[0] += r0;
        acc[1] += x1;
        acc[2] += r2 * delta * delta;
        acc[3] += r0 * y;
        acc[4] += x1 * y;
        acc[5] += r0 * y * y;
        r0 = r1 = r2 = 0.0;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) s_part[k][threadIdx.x] = acc[k];
#pragma unroll
  for (int p = 0; p < kMaxPupils; ++p)
    if (p < npup) s_part[6 + p][threadIdx.x] = ps[p];
  __syncthreads();
  const double a = block_sums<kFPThreads>(s_part, 6 + npup);
  const int k = threadIdx.x / 16;
  if (threadIdx.x % 16 == 0 && k < kMaxSums)
    part[((size_t)b * (N / T) + tile) * kMaxSums + k] = k < 6 + npup ? a : 0.0;
}

// Sum tiles (in a fixed order) and form the measures of measures.py / beam.py.
// A thread's tiles are read whole (112 contiguous bytes each) before the sums
// meet in LDS: 11 us -> 6 us at 512 tiles, where each of the up to 14 sums
// had been a pass over the tiles and an eight-barrier tree.
__global__ void __launch_bounds__(256)
k_moments_finalize(int ntiles, const double* __restrict__ part, const double* __restrict__ chparam,
                   int npup, const int* __restrict__ chan, double* __restrict__ out) {
  const int b = blockIdx.x;
  __shared__ double s_part[kMaxSums][256 + 1];
  __shared__ double S[kMaxSums];
  const int ns = 6 + npup;
  double a[kMaxSums];
#pragma unroll
  for (int k = 0; k < kMaxSums; ++k) a[k] = 0.0;
  for (int t = threadIdx.x; t < ntiles; t += 256) {
    const double* p = part + ((size_t)b * ntiles + t) * kMaxSums;
#pragma unroll
    for (int k = 0; k < kMaxSums; ++k)
      if (k < ns) a[k] += p[k];
  }
#pragma unroll
  for (int k = 0; k < kMaxSums; ++k)
    if (k < ns) s_part[k][threadIdx.x] = a[k];
  __syncthreads();
  const double v = block_sums<256>(s_part, ns);
  if (threadIdx.x % 16 == 0 && threadIdx.x / 16 < kMaxSums)
    S[threadIdx.x / 16] = (int)threadIdx.x / 16 < ns ? v : 0.0;
  __syncthreads();
  if (threadIdx.x != 0) return;
  const int ch = chan ? chan[b] : 0;
  const double delta = chparam[ch * kChParams + 0];
  const double d2 = delta * delta;
  double* o = out + (size_t)b * kMoments;
  const double eta = S[0] * d2, mx = S[1] * d2, my = -S[3] * d2;
  const double mx2 = S[2] * d2, mxy = -S[4] * d2, my2 = S[5] * d2;
  o[0] = eta;
  o[1] = mx;
  o[2] = my;
  o[3] = mx2;
  o[4] = mxy;
  o[5] = my2;
  const double r0 = sqrt(mx * mx + my * my);
  const double cx = mx / r0, sx = my / r0;  // NaN at r0 == 0, as in beam.py:27-30
  o[6] = cx * cx * mx2 + 2.0 * cx * sx * mxy + sx * sx * my2;
  for (int p = 0; p < kMaxPupils; ++p) o[7 + p] = p < npup ? S[6 + p] * d2 : 0.0;
}

__global__ void k_apply_pupil(int n, float2* __restrict__ u, double delta, double rad2, double sx,
                              double sy) {
  const int b = blockIdx.y;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)n * n) return;
  const int r = (int)(idx / n), c = (int)(idx % n);
  if (!in_circle(grid_offset(c, n, delta, sx), grid_offset(r, n, delta, -sy), rad2))
    u[(size_t)b * n * n + idx] = make_float2(0.f, 0.f);
}

// out = u inside the pupil, 0 outside, as a new field: a row's columns inside are
// one interval (circle_cols, the exact predicate), found by one thread per row
// of the block, so the field is read inside the pupil only and nothing is
// tested in float64 per element.  The 8 bytes written per element bound a large
// batch; one field is bound by a block's chain (interval, read, write), so a
// block takes two rows (5.3 us for a 1024^2 field, 10.2 with eight; a copy
// and a pass over it took 16).
constexpr int kPupilRows = 2;
__global__ void __launch_bounds__(256)
k_pupil_output(int n, const float2* __restrict__ u, float2* __restrict__ out, double delta, double rad2, double sx,
               double sy) {
  __shared__ int2 s_pc[kPupilRows];
  const size_t o = (size_t)blockIdx.y * n * n + (size_t)blockIdx.x * kPupilRows * n;
  if (threadIdx.x < kPupilRows) {
    int lo, hi;
    circle_cols(n, delta, grid_offset(blockIdx.x * kPupilRows + threadIdx.x, n, delta, -sy), sx, rad2, lo, hi);
    s_pc[threadIdx.x] = make_int2(lo, hi);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kPupilRows * n / 2; i += 256) {
    const int r = 2 * i >= n, c = 2 * i - r * n;
    const int2 q = s_pc[r];
    pa_f4c v = {0.f, 0.f, 0.f, 0.f};
    if (q.x <= c + 1 && q.y >= c) {
      const pa_f4c w = reinterpret_cast<const pa_f4c*>(u + o)[i];
      if (q.x <= c && c <= q.y) v.x = w.x, v.y = w.y;
      if (q.x <= c + 1 && c + 1 <= q.y) v.z = w.z, v.w = w.w;
    }
    reinterpret_cast<pa_f4c*>(out + o)[i] = v;
  }
}

__global__ void k_expmi(int count, const float* __restrict__ x, float2* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) out[i] = expmi_fast(x[i]);
}

int expmi_eval(int count, const float* x, float2* out, hipStream_t s) {
  hipLaunchKernelGGL(k_expmi, dim3((count + 255) / 256), dim3(256), 0, s, count, x, out);
  return check_launch("expmi");
}

__global__ void k_twiddles(int n, float2* __restrict__ tw) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  double s, c;
  sincospi(2.0 * k / n, &s, &c);
  tw[k] = make_float2((float)c, (float)-s);
}

__global__ void k_outer(int n, float2* __restrict__ out, const float2* __restrict__ gy,
                        const float2* __restrict__ gx) {
  const int b = blockIdx.y;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)n * n) return;
  const int r = (int)(idx / n), c = (int)(idx % n);
  out[(size_t)b * n * n + idx] = cmul(gy[(size_t)b * n + r], gx[(size_t)b * n + c]);
}

__global__ void k_intensity(size_t count, const float2* __restrict__ u, float* __restrict__ out) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= count) return;
  const float2 v = u[idx];
  out[idx] = v.x * v.x + v.y * v.y;
}

int outer(int n, float2* out, const float2* gy, const float2* gx, int batch, hipStream_t s) {
  hipLaunchKernelGGL(k_outer, dim3((n * n + 255) / 256, batch), dim3(256), 0, s, n, out, gy, gx);
  return check_launch("outer");
}

int intensity(long long count, const float2* u, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_intensity, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s, (size_t)count, u, out);
  return check_launch("intensity");
}

template <int N>
static void launch_field_partials(const float2* u, double* part, const double* chparam, const double* pup, int npup,
                                  const double* pup_moments, const int* chan, int batch, hipStream_t s) {
  constexpr int T = Geo<N>::T;
  hipLaunchKernelGGL((k_field_partials<N, T>), dim3(N / T, batch), dim3(kFPThreads), 0, s, u, part, chparam, pup, npup,
                     pup_moments, chan);
}

int field_partials(int n, const float2* u, double* part, const double* chparam, const double* pup,
                   int npup, const double* pup_moments, const int* chan, int batch, hipStream_t s) {
#define C_(NN) \
  case NN: launch_field_partials<NN>(u, part, chparam, pup, npup, pup_moments, chan, batch, s); break;
  switch (n) {
    C_(64) C_(128) C_(256) C_(512) C_(1024) C_(2048) C_(4096)
    default: return set_error(PA_ERR_SIZE, "grid size must be a power of two in [64, 4096]");
  }
#undef C_
  return check_launch("field_partials");
}

int moments_finalize(int n, const double* part, const double* chparam, int npup, const int* chan,
                     double* out, int batch, hipStream_t s) {
  const int T = tile_rows(n);
  if (T <= 0) return T;
  hipLaunchKernelGGL(k_moments_finalize, dim3(batch), dim3(256), 0, s, n / T, part, chparam, npup,
                     chan, out);
  return check_launch("moments_finalize");
}

// ------------------------------------------------------------------ no-allocation moments
// The per-tile partials of pa_field_moments_static live in this file-scope
// device array instead of a caller's buffer.  Each device that runs the entry
// point holds its own copy until the process ends; host code reaches it only
// through the address hipGetSymbolAddress returns for the current device (the
// array's name is a host-side stand-in, not a device address).  Every call on
// a device shares that device's array, so calls that overlap on one device
// (different streams, or threads) race; calls in one stream do not.  Nothing
// needs clearing: k_field_partials writes every partial k_moments_finalize
// reads.
constexpr long long kStaticScratchBytes = 16ll << 20;
static __device__ __align__(256) double scratch[kStaticScratchBytes / sizeof(double)];

// Fields per call.  The limit is that of 8 MiB of partials for tiles of at least
// these heights; the tiles of 256^2 to 1024^2 grids are half as high, for which
// the array has its other half.
int static_max_fields(int n) {
  const int T = tile_rows(n);
  if (T <= 0) return T;
  const int rows = n == 256 ? 16 : n == 512 || n == 1024 ? 8 : T;
  static_assert(Geo<256>::T >= 8 && Geo<512>::T >= 4 && Geo<1024>::T >= 4, "partials fit the array");
  return (int)(kStaticScratchBytes / 2 / ((long long)(n / rows) * kMaxSums * (long long)sizeof(double)));
}

static std::mutex g_scratch_mutex;
static double* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per device.
int static_scratch(double** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_error(PA_ERR_HIP, "field_moments_static: no current HIP device");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return set_error(PA_ERR_HIP, "field_moments_static: hipGetSymbolAddress of the scratch array failed");
    }
    g_scratch_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_scratch_ptr[dev];
  return PA_OK;
}

int field_moments_static(int n, const float2* u, const double* chparam, const double* pup, int npup,
                         const double* pup_moments, const int* chan, double* out, int batch, hipStream_t s) {
  double* part = nullptr;
  int rc = static_scratch(&part);
  if (rc) return rc;
  rc = field_partials(n, u, part, chparam, pup, npup, pup_moments, chan, batch, s);
  if (rc) return rc;
  return moments_finalize(n, part, chparam, npup, chan, out, batch, s);
}

// ------------------------------------------------------------------ ensemble accumulation
// Per-channel Monte Carlo ensembles on the device (simulations/beam.py:35-71;
// simulations/pdt.py:28-48): each realization's finalized moments add to its
// channel's float64 sums of the BeamResult quantities and their squares, and
// each pupil's transmittance to a 64-bin integer histogram over [0, 1].  One
// thread per channel walks the batch in order, so the sums are deterministic
// (no atomics); a channel stops taking beam samples at beam_cap and PDT
// samples at pdt_cap (caps < 0: no limit).  Quantities per sample, in the
// order of PA_ENS_*: eta, mean_x, mean_y, mean_x2, mean_xy, mean_y2,
// mean_x2_r, bw2_x = mean_x^2, bw2_y = mean_y^2, lt2 = 4 mean_x2,
// st2 = lt2 - 4 bw2_x (beam.py:35-47, evaluated with the same roundings).
// Binning follows numpy.histogram(eta, 64, range=(0, 1)): values outside
// [0, 1] (and NaN) are dropped, eta = 1 falls into the last bin, and the bin
// of eta is floor(64 eta) (edges k/64 are exact in float64).
__global__ void __launch_bounds__(256)
k_ensemble_accumulate(int batch, const double* __restrict__ mom, const int* __restrict__ slot_chan, int nchan,
                      int npup, int beam_cap, int pdt_cap, double* __restrict__ acc,
                      long long* __restrict__ counts, unsigned long long* __restrict__ hist) {
  const int ch = blockIdx.x * blockDim.x + threadIdx.x;
  if (ch >= nchan) return;
  double* a = acc + (size_t)ch * 2 * PA_ENS_QUANTITIES;
  long long nb = counts[2 * ch], np_ = counts[2 * ch + 1];
  unsigned long long* h = hist + (size_t)ch * kMaxPupils * PA_PDT_BINS;
  for (int b = 0; b < batch; ++b) {
    if ((slot_chan ? slot_chan[b] : 0) != ch) continue;
    const double* m = mom + (size_t)b * kMoments;
    if (beam_cap < 0 || nb < beam_cap) {
#pragma clang fp contract(off)
      double q[PA_ENS_QUANTITIES];
      for (int k = 0; k < 7; ++k) q[k] = m[k];
      q[7] = m[1] * m[1];
      q[8] = m[2] * m[2];
      q[9] = 4.0 * m[3];
      q[10] = q[9] - 4.0 * q[7];
      for (int k = 0; k < PA_ENS_QUANTITIES; ++k) {
        a[k] += q[k];
        a[PA_ENS_QUANTITIES + k] += q[k] * q[k];
      }
      ++nb;
    }
    if (pdt_cap < 0 || np_ < pdt_cap) {
      for (int p = 0; p < npup; ++p) {
        const double e = m[7 + p];
        if (!(e >= 0.0 && e <= 1.0)) continue;
        int bin = (int)(e * PA_PDT_BINS);
        if (bin == PA_PDT_BINS) bin = PA_PDT_BINS - 1;
        ++h[p * PA_PDT_BINS + bin];
      }
      ++np_;
    }
  }
  counts[2 * ch] = nb;
  counts[2 * ch + 1] = np_;
}

int ensemble_accumulate(int batch, const double* mom, const int* slot_chan, int nchan, int npup, int beam_cap,
                        int pdt_cap, double* acc, long long* counts, unsigned long long* hist, hipStream_t s) {
  hipLaunchKernelGGL(k_ensemble_accumulate, dim3((nchan + 255) / 256), dim3(256), 0, s, batch, mom, slot_chan,
                     nchan, npup, beam_cap, pdt_cap, acc, counts, hist);
  return check_launch("ensemble_accumulate");
}

int apply_pupil(int n, float2* u, double delta, double radius, double sx, double sy, int batch,
                hipStream_t s) {
  hipLaunchKernelGGL(k_apply_pupil, dim3((n * n + 255) / 256, batch), dim3(256), 0, s, n, u, delta,
                     radius * radius, sx, sy);
  return check_launch("apply_pupil");
}

int pupil_output(int n, const float2* u, float2* out, double delta, double radius, double sx, double sy, int batch,
                 hipStream_t s) {
  hipLaunchKernelGGL(k_pupil_output, dim3(n / kPupilRows, batch), dim3(256), 0, s, n, u, out, delta, radius * radius, sx,
                     sy);
  return check_launch("pupil_output");
}

// ------------------------------------------------------------------ structure function
// Row structure function of a screen (theory/phase_screens/sf.py:4-8 averaged
// over rows as in simulations/structure_function.py:11-12):
//   D[r - 1] = (1 / rows) sum_rows (1 / (n - r)) sum_{c < n - r} (phi[c] - phi[c + r])^2.
// Per (row, lag) the squares are summed in float32 over four interleaved
// accumulators (the reference's own arithmetic is float32; columns past the last
// whole quad go to the first one), then in float64 over rows.
//
// k_sf_partials: one block per kSFRows rows of element b, the rows in LDS.
// The N^3 / 2 squared differences bound it (two vector operations each, 27 us
// at 1024^2), so a thread takes the four lags 4 g .. 4 g + 3 at once: for each
// quad of columns it reads one new quad of the shifted row (the seven values
// the four lags need slide through two register quads) and one quad that the
// whole wave shares, two 16-byte LDS reads for 16 differences instead of two
// dword reads for each.  Lag group g has n / 4 - g quads, so a thread takes the
// groups g and n / 4 - 1 - g in turn and all threads have equal work.
// k_sf_finalize adds the row groups with 16 waves per 64 lags and divides by
// (n - r) n.
// Measured at 1024^2, one screen: 186 us (partials) and 68 us (finalize) with one
// lag per thread and one thread per lag, 37 and 5 us so.
constexpr int kSFRows = 4;
constexpr int kSFThreads = 512;
typedef float pa_f4u __attribute__((ext_vector_type(4), aligned(4)));   // screens need no more than float alignment

template <int N>
__global__ void __launch_bounds__(kSFThreads)
k_sf_partials(const float* __restrict__ phi, double* __restrict__ part) {
  constexpr int Q = N / 4;                       // quads per row = lag groups
  __shared__ float4 s_row[kSFRows * Q];
  __shared__ float4 s_sum[kSFRows * Q];          // per row, lags 4 g .. 4 g + 3
  const int b = blockIdx.y, g0 = blockIdx.x;
  const pa_f4u* src = reinterpret_cast<const pa_f4u*>(phi + ((size_t)b * N + (size_t)g0 * kSFRows) * N);
  for (int i = threadIdx.x; i < kSFRows * Q; i += kSFThreads) {
    const pa_f4u v = src[i];
    s_row[i] = make_float4(v.x, v.y, v.z, v.w);
  }
  __syncthreads();
  for (int task = threadIdx.x; task < kSFRows * Q / 2; task += kSFThreads) {
    const int q = task / (Q / 2), p = task % (Q / 2);
    const float4* row = s_row + q * Q;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int g = side ? Q - 1 - p : p;
      float acc[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
      float4 lo = row[g];
      const int kc = Q - 1 - g;                  // whole quads of every lag of the group
#pragma unroll 2
      for (int k = 0; k < kc; ++k) {
        const float4 x = row[k], hi = row[k + g + 1];
        const float xv[4] = {x.x, x.y, x.z, x.w};
        const float w[7] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float d = xv[j] - w[i + j];
            acc[i][j] = fmaf(d, d, acc[i][j]);
          }
        lo = hi;
      }
      // the last quad: whole for lag 4 g, and 3, 2, 1 columns of lags 4 g + 1 .. 3
      const float4 x = row[kc];
      const float xv[4] = {x.x, x.y, x.z, x.w};
      const float w[4] = {lo.x, lo.y, lo.z, lo.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j + i < 4; ++j) {
          const float d = xv[j] - w[i + j];
          float& a = acc[i][i ? 0 : j];
          a = fmaf(d, d, a);
        }
      float4 v;
      v.x = (acc[0][0] + acc[0][1]) + (acc[0][2] + acc[0][3]);
      v.y = (acc[1][0] + acc[1][1]) + (acc[1][2] + acc[1][3]);
      v.z = (acc[2][0] + acc[2][1]) + (acc[2][2] + acc[2][3]);
      v.w = (acc[3][0] + acc[3][1]) + (acc[3][2] + acc[3][3]);
      s_sum[q * Q + g] = v;
    }
  }
  __syncthreads();
  const float* sum = reinterpret_cast<const float*>(s_sum);
  double* dst = part + ((size_t)b * (N / kSFRows) + g0) * (N - 1);
  for (int r = 1 + threadIdx.x; r < N; r += kSFThreads) {
    double a = 0.0;
#pragma unroll
    for (int q = 0; q < kSFRows; ++q) a += (double)sum[q * N + r];
    dst[r - 1] = a;
  }
}

__global__ void __launch_bounds__(1024)
k_sf_finalize(int n, const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double s[16][64];
  const int b = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = 1 + blockIdx.x * 64 + lane;
  const int groups = n / kSFRows;
  const double* p = part + (size_t)b * groups * (n - 1) + (r - 1);
  double v = 0.0;
  if (r < n) {
#pragma unroll 4
    for (int g = wave; g < groups; g += 16) v += p[(size_t)g * (n - 1)];
  }
  s[wave][lane] = v;
  __syncthreads();
  if (wave || r >= n) return;
  for (int w = 1; w < 16; ++w) v += s[w][lane];
  out[(size_t)b * (n - 1) + r - 1] = v / ((double)(n - r) * n);
}

long long sf_scratch_bytes(int n, int batch) {
  return (long long)batch * (n / kSFRows) * (n - 1) * (long long)sizeof(double);
}

template <int N>
static void launch_sf_partials(const float* phi, double* part, int batch, hipStream_t s) {
  hipLaunchKernelGGL(k_sf_partials<N>, dim3(N / kSFRows, batch), dim3(kSFThreads), 0, s, phi, part);
}

int structure_function(int n, const float* phi, double* part, double* out, int batch, hipStream_t s) {
  switch (n) {
    case 64: launch_sf_partials<64>(phi, part, batch, s); break;
    case 128: launch_sf_partials<128>(phi, part, batch, s); break;
    case 256: launch_sf_partials<256>(phi, part, batch, s); break;
    case 512: launch_sf_partials<512>(phi, part, batch, s); break;
    case 1024: launch_sf_partials<1024>(phi, part, batch, s); break;
    case 2048: launch_sf_partials<2048>(phi, part, batch, s); break;
    case 4096: launch_sf_partials<4096>(phi, part, batch, s); break;
    default: return set_error(PA_ERR_SIZE, "grid size must be a power of two in [64, 4096]");
  }
  hipLaunchKernelGGL(k_sf_finalize, dim3((n - 1 + 63) / 64, batch), dim3(1024), 0, s, n, part, out);
  return check_launch("structure_function");
}

int fill_twiddles(int n, float2* tw, hipStream_t s) {
  hipLaunchKernelGGL(k_twiddles, dim3((n + 255) / 256), dim3(256), 0, s, n, tw);
  return check_launch("twiddles");
}

}  // namespace pa
