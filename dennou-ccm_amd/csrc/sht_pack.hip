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

// Small calls: one thread per (canonical k, field), field fastest: canonical writes coalesce
__global__ void spml_to_canon_each_kernel(const double *__restrict__ wa, double *__restrict__ spec,
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

// Small calls: one thread per (field, l), l fastest: SPML-layout writes coalesce
__global__ void canon_to_spml_each_kernel(const double *__restrict__ spec, double *__restrict__ wa,
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

// SPML packing <-> canonical spectra: a workgroup transposes the degree n of
// kPackFields fields through LDS.  On the SPML side a field's degree is one
// run of 2n + 1 reals (l = n(n+1) + m, m = -n..n); on the canonical side each
// (m, n) row holds the fields' complex values next to each other, 128 bytes of
// them per group.  A thread per element of one side has to gather or scatter
// single values on the other (the kernels above, for small calls: pack_each).
// T85, 97 fields (5.7 + 5.8 MB), back to back: to canonical 7.8 -> 4.4 us, to
// SPML 9.8 -> 4.0 us.
// The groups of one degree run on one XCD, so the parts of the lines that
// neighbouring groups share meet in its L2; degrees are dealt to the XCDs in
// turn, longest first.
constexpr int kPackFields = 8;
// row pitch of the LDS tile [field][2n + 1]: 8 past a multiple of 16 doubles,
// so 8 fields x 8 consecutive m read without bank conflicts
__host__ __device__ inline int pack_pitch(int N) { return roundup(2 * N + 1, 16) + 8; }

struct PackTile {
  int n, f0, nf;  // degree, first field, fields of the group
  __device__ __forceinline__ bool at(unsigned b, int N, int nfields) {
    const unsigned ng = ((unsigned)nfields + kPackFields - 1) / kPackFields, j = b >> 3;
    n = N - (int)((j / ng) * 8 + (b & 7));
    f0 = (int)(j % ng) * kPackFields;
    nf = nfields - f0 < kPackFields ? nfields - f0 : kPackFields;
    return n >= 0;
  }
};
inline unsigned pack_tiles(int N, int nf) {
  return 8u * ((N + 8) / 8) * (((unsigned)nf + kPackFields - 1) / kPackFields);
}
// workgroups of a launch (a multiple of 8): a few fields of huge batches take several tiles each
inline unsigned pack_blocks(unsigned tiles) { return tiles < (1u << 20) ? tiles : 1u << 20; }

__global__ __launch_bounds__(256) void spml_to_canon_kernel(const double *__restrict__ wa,
                                                            double *__restrict__ spec, int N, int nf,
                                                            unsigned tiles) {
  extern __shared__ double tile[];
  for (unsigned blk = blockIdx.x; blk < tiles; blk += gridDim.x) {
    PackTile pt;
    if (!pt.at(blk, N, nf)) continue;
    const int n = pt.n, cnt = 2 * n + 1, pitch = pack_pitch(N), wave = wave_id(), lane = threadIdx.x & 63;
    const size_t L = (size_t)(N + 1) * (N + 1);
    // wave w reads fields w and w + 4, two runs of 64 of each at a time
    const int fa = wave, fb = wave + 4;
    const double *__restrict__ wn = wa + (size_t)pt.f0 * L + (size_t)n * n;
    const double *__restrict__ a = wn + (fa < pt.nf ? fa : 0) * L, *__restrict__ b = wn + (fb < pt.nf ? fb : 0) * L;
    for (int l = lane; l < cnt; l += 128) {
      const int l2 = l + 64 < cnt ? l + 64 : l;
      const double a0 = a[l], b0 = b[l], a1 = a[l2], b1 = b[l2];
      tile[fa * pitch + l] = a0;
      tile[fb * pitch + l] = b0;
      tile[fa * pitch + l2] = a1;
      tile[fb * pitch + l2] = b1;
    }
    __syncthreads();
    const int f = threadIdx.x & (kPackFields - 1);
    double *__restrict__ out = spec + 2 * (pt.f0 + f);  // 8-byte aligned, as the caller's array
    for (int m = threadIdx.x / kPackFields; f < pt.nf && m <= n; m += 256 / kPackFields) {
      const double re = tile[f * pitch + n + m], im = tile[f * pitch + n - m];
      double *__restrict__ o = out + (size_t)(coef_off(N, m) + n - m) * 2 * nf;
      o[0] = m == 0 ? re : re / kSqrt2;
      o[1] = m == 0 ? 0.0 : -im / kSqrt2;
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void canon_to_spml_kernel(const double *__restrict__ spec,
                                                            double *__restrict__ wa, int N, int nf,
                                                            unsigned tiles) {
  extern __shared__ double tile[];
  for (unsigned blk = blockIdx.x; blk < tiles; blk += gridDim.x) {
    PackTile pt;
    if (!pt.at(blk, N, nf)) continue;
    const int n = pt.n, cnt = 2 * n + 1, pitch = pack_pitch(N), wave = wave_id(), lane = threadIdx.x & 63;
    const int f = threadIdx.x & (kPackFields - 1), fc = f < pt.nf ? f : 0;
    const double *__restrict__ in = spec + 2 * (pt.f0 + fc);  // 8-byte aligned, as the caller's array
    constexpr int kRows = 256 / kPackFields;  // m rows the block reads at once
    for (int m0 = threadIdx.x / kPackFields; m0 <= n; m0 += 2 * kRows) {
      const int m1 = m0 + kRows <= n ? m0 + kRows : m0;
      const double *__restrict__ i0 = in + (size_t)(coef_off(N, m0) + n - m0) * 2 * nf;
      const double *__restrict__ i1 = in + (size_t)(coef_off(N, m1) + n - m1) * 2 * nf;
      const double2 v0 = make_double2(i0[0], i0[1]), v1 = make_double2(i1[0], i1[1]);
      // m = 0 writes its one slot with both stores, the real part last
      tile[f * pitch + n - m0] = -kSqrt2 * v0.y;
      tile[f * pitch + n + m0] = m0 == 0 ? v0.x : kSqrt2 * v0.x;
      tile[f * pitch + n - m1] = -kSqrt2 * v1.y;
      tile[f * pitch + n + m1] = m1 == 0 ? v1.x : kSqrt2 * v1.x;
    }
    __syncthreads();
    const size_t L = (size_t)(N + 1) * (N + 1);
    for (int g = wave; g < pt.nf; g += 4) {
      double *__restrict__ o = wa + (size_t)(pt.f0 + g) * L + (size_t)n * n;
      for (int l = lane; l < cnt; l += 64) o[l] = tile[g * pitch + l];
    }
    __syncthreads();
  }
}

// one block per field: (1/4pi) sum_ij (2pi/im) w_j f_ij.  One CU reads a whole
// field, so the kernel is bound by what that CU has in flight and by its load
// instructions: every thread issues kAvrAhead 16-byte loads before it adds the
// first (W = 2 values; W = 1 for a grid that is only 8-byte aligned), and the
// block is as wide as the field allows (avr_threads).  LONG, for fields of more
// than one such round of a full block: the next round's loads are in flight
// while one is added, and the row weights come from LDS instead of a second
// load per pair; a thread adds the same values in the same order either way.
// 12 fields of 256 x 128: 6.1 -> 4.9 us (37.9 with 256 threads and one load at a
// time), 97 fields 7.1 -> 6.6, one field of 512 x 256 16.9 -> 10.4; 8-byte
// loads 6.9 us at 12 fields.  Fields of one round gain nothing from it and pay
// the barrier (128 x 64, 26 fields 3.3 against 3.6 us).  A pair never straddles a
// row: im is even.
constexpr int kAvrAhead = 8, kAvrMaxRows = 512;
template <int W, bool LONG>
__global__ __launch_bounds__(1024) void avr_kernel(const double *__restrict__ grid,
                                                   const double *__restrict__ w,
                                                   double *__restrict__ avg, int im, int lim, int n) {
  typedef double vec __attribute__((ext_vector_type(W)));
  const int f = blockIdx.x, step = blockDim.x * W;
  const double *__restrict__ g = grid + (size_t)f * n;
  double acc = 0.0;
  auto load = [&](int t0, vec (&v)[kAvrAhead]) {
#pragma unroll
    for (int q = 0; q < kAvrAhead; ++q) {
      const int t = t0 + q * step;
      v[q] = *reinterpret_cast<const vec *>(g + (t < n ? t : 0));  // past the end: a valid address, not added
    }
  };
  auto add = [&](int t0, const vec (&v)[kAvrAhead], auto weight) {
#pragma unroll
    for (int q = 0; q < kAvrAhead; ++q)
      if (t0 + q * step < n)
#pragma unroll
        for (int i = 0; i < W; ++i) acc += weight(q) * v[q][i];
  };
  int t0 = threadIdx.x * W;
  if constexpr (LONG) {
    __shared__ double ws[kAvrMaxRows];
    vec a[kAvrAhead], b[kAvrAhead];
    load(t0, a);
    for (int j = threadIdx.x; j < n >> lim; j += blockDim.x) ws[j] = w[j];
    __syncthreads();
    for (; t0 < n; t0 += 2 * kAvrAhead * step) {
      const int t1 = t0 + kAvrAhead * step, t2 = t1 + kAvrAhead * step;
      load(t1, b);
      add(t0, a, [&](int q) { return ws[(t0 + q * step) >> lim]; });
      if (t2 < n) load(t2, a);
      add(t1, b, [&](int q) { return ws[(t1 + q * step) >> lim]; });
    }
  } else {
    for (; t0 < n; t0 += kAvrAhead * step) {
      vec v[kAvrAhead];
      double wj[kAvrAhead];
      load(t0, v);
#pragma unroll
      for (int q = 0; q < kAvrAhead; ++q) wj[q] = w[(t0 + q * step < n ? t0 + q * step : t0) >> lim];
      add(t0, v, [&](int q) { return wj[q]; });
    }
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
  __shared__ double red[16];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  // the waves' sums pairwise: added in a row, their roundings are half as large
  // again as all others together (256 x 128, rms error 1.2e-16 against 0.9e-16)
  if (threadIdx.x < 16) {
    acc = threadIdx.x < blockDim.x >> 6 ? red[threadIdx.x] : 0.0;
#pragma unroll
    for (int s = 8; s > 0; s >>= 1) acc += __shfl_xor(acc, s);
    if (threadIdx.x == 0) avg[f] = acc / (2.0 * im);
  }
}
// a wave for each 64 x 2 kAvrAhead points, up to 16 waves
inline int avr_threads(int n) {
  const int t = roundup((n + 2 * kAvrAhead - 1) / (2 * kAvrAhead), 64);
  return t < 1024 ? t : 1024;
}

// out = (-n(n+1))^power in on the canonical rows, one complex value per thread.
// Every block makes the factors of all degrees once (LDS) while its loads are
// in flight, and finds a value's degree in closed form (lapla_degree).  T85, 97
// fields (5.8 MB each way), back to back: 13.8 -> 3.9 us with a search for m
// and a power per value before (four values per thread: 5.3 us, and slower at
// every size up to 11 M values).
// degree of canonical row k: off(m) = m (2N + 3 - m) / 2, so the largest m with
// off(m) <= k is the floor of the smaller root of m^2 - (2N + 3) m + 2k; the
// FP32 root is within one of it (all terms are below 2^24) and is corrected
__device__ __forceinline__ int lapla_degree(int N, int k) {
  const float b = (float)(2 * N + 3);
  int m = (int)(0.5f * (b - sqrtf(b * b - 8.0f * (float)k)));
  m = m < 0 ? 0 : m > N ? N : m;
  auto off = [&](int x) { return (x * (2 * N + 3 - x)) >> 1; };
  while (m > 0 && off(m) > k) --m;
  while (m < N && off(m + 1) <= k) ++m;
  return m + k - off(m);
}
__global__ __launch_bounds__(256) void lapla_kernel(const double2 *in, double2 *out, int N, int nf,
                                                    int power, int64_t total) {
  __shared__ double fac[256];  // N <= 255
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const double2 v = t < total ? in[t] : make_double2(0.0, 0.0);
  if ((int)threadIdx.x <= N) {
    const int n = threadIdx.x;
    const double e = -(double)n * (n + 1);
    double x = 1.0;
    if (power < 0 && n == 0) {
      x = 0.0;
    } else {
      const int ap = power < 0 ? -power : power;
      for (int i = 0; i < ap; ++i) x = power < 0 ? x / e : x * e;
    }
    fac[n] = x;
  }
  __syncthreads();
  if (t >= total) return;
  // 32-bit division where it suffices
  const int k = total <= UINT32_MAX ? (int)((uint32_t)t / (uint32_t)nf) : (int)(t / nf);
  const double x = fac[lapla_degree(N, k)];
  out[t] = make_double2(x * v.x, x * v.y);
}

// Which kernel converts a call: one thread per value, or the tiles.  The tiles
// pay where there are values enough to be bound by lines touched; a tile of few
// fields leaves most of its lanes idle, one of a short degree (below 32) too, and
// degrees above 63 take several rounds of rows in few workgroups.  Back to back,
// per value / tiles, us: to canonical T85 1 field 2.27 / 3.26, 16 fields 2.72 / 2.83,
// 32 fields 3.23 / 2.99; T42 8 fields equal, 64 fields 2.75 / 2.58; T170 5 fields 2.89 /
// 3.51, 12 fields 3.80 / 3.63; T21 776 fields 3.91 / 4.87, 1500 fields equal; to SPML
// T85 1 field 2.05 / 2.42, 24 fields 2.69 / 2.79, 32 fields 3.00 / 2.85; T42 26 fields
// 2.20 / 2.36, 79 fields 2.55 / 2.52.
inline bool pack_each(const Plan &p, int nf, bool to_canon) {
  const int64_t values = (int64_t)p.K * nf;
  if (p.N < 32 || nf < kPackFields) return values <= 200000;
  return p.N < 64 ? !to_canon && values <= 65536 : values <= (to_canon ? 65536 : 100000);
}

}  // namespace

int launch_spec_lapla(const Plan &p, const double *in, double *out, int power, int nf,
                      hipStream_t s) {
  const int64_t n = (int64_t)p.K * nf;
  lapla_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
      reinterpret_cast<const double2 *>(in), reinterpret_cast<double2 *>(out), p.N, nf, power, n);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_spml_to_canon(const Plan &p, const double *wa, double *spec, int nf, hipStream_t s) {
  if (pack_each(p, nf, true)) {
    spml_to_canon_each_kernel<<<(unsigned)(((int64_t)p.K * nf + 255) / 256), 256, 0, s>>>(wa, spec, p.N, nf);
  } else {
    const unsigned tiles = pack_tiles(p.N, nf);
    spml_to_canon_kernel<<<pack_blocks(tiles), 256, sizeof(double) * kPackFields * pack_pitch(p.N), s>>>(
        wa, spec, p.N, nf, tiles);
  }
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_canon_to_spml(const Plan &p, const double *spec, double *wa, int nf, hipStream_t s) {
  if (pack_each(p, nf, false)) {
    canon_to_spml_each_kernel<<<(unsigned)(((int64_t)(p.N + 1) * (p.N + 1) * nf + 255) / 256), 256, 0, s>>>(
        spec, wa, p.N, nf);
  } else {
    const unsigned tiles = pack_tiles(p.N, nf);
    canon_to_spml_kernel<<<pack_blocks(tiles), 256, sizeof(double) * kPackFields * pack_pitch(p.N), s>>>(
        spec, wa, p.N, nf, tiles);
  }
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

int launch_avr_lonlat(const Plan &p, const double *grid, double *avg, int nf, hipStream_t s) {
  const int n = p.im * p.jm;
  const bool two = ((uintptr_t)grid & 15) == 0, lng = n > 2 * kAvrAhead * 1024;
  const auto kern = two ? (lng ? avr_kernel<2, true> : avr_kernel<2, false>)
                        : (lng ? avr_kernel<1, true> : avr_kernel<1, false>);
  kern<<<nf, avr_threads(n), 0, s>>>(grid, p.w, avg, p.im, __builtin_ctz(p.im), n);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

}  // namespace sht
