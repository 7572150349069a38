// sht_pack.hip -- spectral layout conversion between SPML's real (N+1)^2
// packing (Fortran wa((N+1)**2, k), index l = n(n+1)+m+1 of SPML l_nm) and the
// canonical complex m-major layout the Legendre GEMMs read, plus the global
// mean AvrLonLat_xy (atm/dccm_atm_mod.f90:668-669, :774) and the diagonal
// spectral operators (SPML wa_Lapla_wa / wa_LaplaInv_wa and their powers, the
// hyperdiffusion of DCPAM's dynamics namelist, HDOrder in
// exp/APEI07Couple/common/dcpam/dcpam_APEI07Couple_T21L16.conf:205-230).
#include "sht_internal.h"

namespace sht {
namespace {

constexpr double kSqrt2 = 1.41421356237309504880;

// one thread per (canonical k, field), field fastest: canonical writes coalesce
__global__ void spml_to_canon_kernel(const double *__restrict__ wa, double *__restrict__ spec,
                                     int N, int nf) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int K = (N + 1) * (N + 2) / 2;
  if (t >= (int64_t)K * nf) return;
  const int f = (int)(t % nf);
  const int k = (int)(t / nf);
  // invert k = off(m) + n - m: off(m) = m (2N + 3 - m) / 2, so the largest m
  // with off(m) <= k is the floor of the smaller root of m^2 - (2N+3) m + 2k,
  // corrected by a step where the square root rounds across an integer
  const double b = 2.0 * N + 3.0;
  int m = (int)floor(0.5 * (b - sqrt(b * b - 8.0 * (double)k)));
  m = m < 0 ? 0 : m > N ? N : m;
  while (m > 0 && coef_off(N, m) > k) --m;
  while (m < N && coef_off(N, m + 1) <= k) ++m;
  const int n = m + (k - (int)coef_off(N, m));
  const double *w = wa + (size_t)f * (N + 1) * (N + 1);
  double re, im;
  if (m == 0) {
    re = w[n * (n + 1)];
    im = 0.0;
  } else {
    re = w[n * (n + 1) + m] / kSqrt2;
    im = -w[n * (n + 1) - m] / kSqrt2;
  }
  spec[2 * t] = re;
  spec[2 * t + 1] = im;
}

// one thread per (field, l), l fastest: SPML-layout writes coalesce
__global__ void canon_to_spml_kernel(const double *__restrict__ spec, double *__restrict__ wa,
                                     int N, int nf) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int L = (N + 1) * (N + 1);
  if (t >= (int64_t)L * nf) return;
  const int l = (int)(t % L);
  const int f = (int)(t / L);
  int n = (int)sqrt((double)l);
  while (n * n > l) --n;
  while ((n + 1) * (n + 1) <= l) ++n;
  const int m = l - n * (n + 1);
  const int am = m < 0 ? -m : m;
  const double *s = spec + ((size_t)(coef_off(N, am) + n - am) * nf + f) * 2;
  double v;
  if (m == 0) v = s[0];
  else if (m > 0) v = kSqrt2 * s[0];
  else v = -kSqrt2 * s[1];
  wa[t] = v;
}

// one block per field: (1/4pi) sum_ij (2pi/im) w_j f_ij.  One CU reads a whole
// field, so the kernel is bound by what that CU has in flight: every thread
// issues kAvrAhead 16-byte loads before it adds the first (W = 2 values; W = 1
// for a grid that is only 8-byte aligned), and the block is as wide as the
// field allows (avr_threads).  12 fields of 256 x 128: 37.9 -> 5.7 us (256
// threads, one load at a time before); with 8-byte loads 9.8 us.  A pair never
// straddles a row: im is even.
constexpr int kAvrAhead = 8;
template <int W>
__global__ __launch_bounds__(1024) void avr_kernel(const double *__restrict__ grid,
                                                   const double *__restrict__ w,
                                                   double *__restrict__ avg, int im, int lim, int n) {
  typedef double vec __attribute__((ext_vector_type(W)));
  const int f = blockIdx.x, step = blockDim.x * W;
  const double *__restrict__ g = grid + (size_t)f * n;
  double acc = 0.0;
  for (int t0 = threadIdx.x * W; t0 < n; t0 += kAvrAhead * step) {
    vec v[kAvrAhead];
    double wj[kAvrAhead];
#pragma unroll
    for (int q = 0; q < kAvrAhead; ++q) {
      const int t = t0 + q * step, c = t < n ? t : t0;  // past the end: a valid address, not added
      v[q] = *reinterpret_cast<const vec *>(g + c);
      wj[q] = w[c >> lim];
    }
#pragma unroll
    for (int q = 0; q < kAvrAhead; ++q)
      if (t0 + q * step < n)
#pragma unroll
        for (int i = 0; i < W; ++i) acc += wj[q] * v[q][i];
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
  __shared__ double red[16];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < (int)blockDim.x >> 6; ++q) acc += red[q];
    avg[f] = acc / (2.0 * im);
  }
}
// a wave for each 64 x 2 kAvrAhead points, up to 16 waves
inline int avr_threads(int n) {
  const int t = roundup((n + 2 * kAvrAhead - 1) / (2 * kAvrAhead), 64);
  return t < 1024 ? t : 1024;
}

// one thread per (canonical k, field) complex pair: out = (-n(n+1))^power in
__global__ void lapla_kernel(const double2 *__restrict__ in, double2 *__restrict__ out, int N,
                             int nf, int power) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int K = (N + 1) * (N + 2) / 2;
  if (t >= (int64_t)K * nf) return;
  const int k = (int)(t / nf);
  int m = 0;
  while (m < N && coef_off(N, m + 1) <= k) ++m;
  const int n = m + (k - (int)coef_off(N, m));
  const double e = -(double)n * (n + 1);
  double fac = 1.0;
  if (power < 0 && n == 0) {
    fac = 0.0;
  } else {
    const int ap = power < 0 ? -power : power;
    for (int i = 0; i < ap; ++i) fac = power < 0 ? fac / e : fac * e;
  }
  const double2 v = in[t];
  out[t] = make_double2(fac * v.x, fac * v.y);
}

}  // namespace

int launch_spec_lapla(const Plan &p, const double *in, double *out, int power, int nf,
                      hipStream_t s) {
  const int64_t n = (int64_t)p.K * nf;
  lapla_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
      reinterpret_cast<const double2 *>(in), reinterpret_cast<double2 *>(out), p.N, nf, power);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_spml_to_canon(const Plan &p, const double *wa, double *spec, int nf, hipStream_t s) {
  const int64_t n = (int64_t)p.K * nf;
  spml_to_canon_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(wa, spec, p.N, nf);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_canon_to_spml(const Plan &p, const double *spec, double *wa, int nf, hipStream_t s) {
  const int64_t n = (int64_t)(p.N + 1) * (p.N + 1) * nf;
  canon_to_spml_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(spec, wa, p.N, nf);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_avr_lonlat(const Plan &p, const double *grid, double *avg, int nf, hipStream_t s) {
  const int n = p.im * p.jm;
  const auto kern = ((uintptr_t)grid & 15) == 0 ? avr_kernel<2> : avr_kernel<1>;
  kern<<<nf, avr_threads(n), 0, s>>>(grid, p.w, avg, p.im, __builtin_ctz(p.im), n);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

}  // namespace sht
