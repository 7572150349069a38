// sht_legendre.hip -- the Gauss-Legendre step in FP64 on the matrix cores.
//
// Per zonal wavenumber m the transform is a pair of small GEMMs, one per
// equatorial parity of n - m (ISPACK's symmetric/antisymmetric Legendre
// transform behind SPML wa_xya / xya_wa):
//   inverse  E[p][c] = sum_k Pt_{m+2k}^m(mu_p)   s[m+2k][c]
//            O[p][c] = sum_k Pt_{m+2k+1}^m(mu_p) s[m+2k+1][c]
//   forward  s[m+2k+par][c] = sum_p (w_p/2) Pt^m(mu_p) SA_par[p][c]
// where c runs over 2 * nfield real columns (complex spectra, fields
// innermost), so levels x fields are the GEMMs' batch dimension.
//
// Each workgroup computes one (m, 16-column tile) with
// v_mfma_f64_16x16x4f64: A = table fragment (16 rows x 4; lane l holds row
// l%16, k l/16), B = data fragment (4 x 16 columns; lane l holds k l/16,
// column l%16), D = 16 x 16 accumulators, 4 doubles per lane: item v of lane l
// is row 4v + l/16, column l%16 (measured on gfx950 with a one-hot lane
// probe).  All global fragments are 128-byte runs.
// Work per m shrinks with m (N - m + 1 degrees), so tiles are ordered heaviest
// first and dealt to the XCDs round robin in launch order (consecutive
// workgroups go to consecutive XCDs), which gives every XCD an equal share of
// heavy and light m; contiguous ranges per XCD would give the first XCD twice
// the average work.
#include "sht_internal.h"

namespace sht {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma_f64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kWaves = 4;   // wavefronts per workgroup, splitting the GEMM's K dimension
constexpr int kSteps = 4;   // K-steps (of 4) per wave whose fragments are loaded at once

// Inverse: spec -> four (tab 0, value table) and/or four2 (tab 1, derivative
// table, written with the parity slots swapped because (1-mu^2) dPt/dmu has the
// opposite equatorial parity to Pt).
// Workgroup = one (m, 16-column tile); wave w takes the K-steps w, w+4, ...,
// issues all their table and spectral fragments at once, runs its MFMAs over
// RT row tiles (16 latitude pairs each), and the four partial sums are added
// in FP64 through LDS.
template <int RT, bool NT>
__global__ __launch_bounds__(256) void leg_inv_f64_kernel(
    const double *__restrict__ spec, double *__restrict__ four, double *__restrict__ four2,
    const double *__restrict__ Pinv, const double *__restrict__ Hinv,
    const int *__restrict__ poff, const int *__restrict__ mlist, int mlen, int N, int P2, int P2p,
    int ncol, int nct, int tab0, int ntab, FourGeom geo) {
  extern __shared__ double red[]; // [kWaves][RT][4][64]
  int m, t;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, ntab * nct, m, t)) return;
  const int ct = t % nct;
  const int tab = tab0 + t / nct;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KP = (ke + 3) & ~3, nsteps = KP >> 2;
  const double *__restrict__ T = (tab ? Hinv : Pinv) + poff[m];
  double *__restrict__ out = tab ? four2 : four;
  const int se = tab ? 1 : 0, so = 1 - se;
  const double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol;
  const int col = ct * 16 + r16;
  const bool cok = col < ncol;

  for (int rt0 = 0; rt0 < P2p / 16; rt0 += RT) {
    // both parities' fragments are issued in the same round of loads
    d4 acc[2][RT];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int r = 0; r < RT; ++r) acc[q][r] = d4{0.0, 0.0, 0.0, 0.0};
    const double *__restrict__ Tp = T + rt0 * 16 + r16;
    const double *__restrict__ sp = sm + col;
    for (int j0 = 0; wave + kWaves * j0 < nsteps; j0 += kSteps) {
      double a[2][kSteps][RT], bv[2][kSteps];
#pragma unroll
      for (int j = 0; j < kSteps; ++j) {
        const int st = wave + kWaves * (j0 + j), k = st * 4 + kq;
        const bool ok = st < nsteps;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          bv[q][j] = (ok && cok && k < (q ? ko : ke)) ? sp[(size_t)(2 * k + q) * ncol] : 0.0;
#pragma unroll
          for (int r = 0; r < RT; ++r)
            a[q][j][r] = ok ? Tp[(size_t)(q * KP + k) * P2p + r * 16] : 0.0;
        }
      }
#pragma unroll
      for (int j = 0; j < kSteps; ++j)
        if (wave + kWaves * (j0 + j) < nsteps)
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[q][r] = mfma_f64(a[q][j][r], bv[q][j], acc[q][r]);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[((wave * RT + r) * 4 + i) * 64 + lane] = acc[q][r][i];
      __syncthreads();
      const int slot = q ? so : se;
      for (int e = threadIdx.x; e < RT * 256; e += 256) {
        const double v = red[e] + red[e + RT * 256] + red[e + 2 * RT * 256] + red[e + 3 * RT * 256];
        const int ln = e & 63, ri = e >> 6, i = ri & 3, r = ri >> 2;
        const int p = (rt0 + r) * 16 + i * 4 + (ln >> 4), c = ct * 16 + (ln & 15);
        if (p < P2 && c < ncol) put_four<NT>(out + geo.at(p, m, slot, c), v);
      }
      __syncthreads();
    }
  }
}

// Forward: four (S, A halves) -> spec.  Workgroup = one (m, 16-column tile);
// wave w takes the latitude-pair steps w, w+4, ... (4 pairs each) of the
// quadrature, the partial sums over its pairs meet in LDS and are added in
// FP64.  MAXRT = row tiles of 16 degrees per parity at m = 0.
template <int MAXRT>
__global__ __launch_bounds__(256) void leg_fwd_f64_kernel(const double *__restrict__ four,
                                                          double *__restrict__ spec,
                                                          const double *__restrict__ Pfwd,
                                                          const int *__restrict__ poff,
                                                          const int *__restrict__ mlist, int mlen,
                                                          int N, int P2, int P2p, int ncol, int nct,
                                                          FourGeom geo) {
  extern __shared__ double red[]; // [kWaves][MAXRT][4][64]
  int m, ct;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, nct, m, ct)) return;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int nn = N - m + 1, ke = (nn + 1) >> 1;
  const int KR = (ke + 15) & ~15, nrt = KR >> 4;
  const int nsteps = P2p >> 2;
  const int col = ct * 16 + r16;
  const bool cok = col < ncol;
  double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol;
  const int kcnt[2] = {ke, nn >> 1};
  d4 acc[2][MAXRT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < MAXRT; ++r) acc[q][r] = d4{0.0, 0.0, 0.0, 0.0};
  const double *__restrict__ W = Pfwd + poff[m] + r16;
  const int csafe = cok ? col : 0;
  // Loads go to clamped, always-valid addresses and are masked afterwards, so
  // the compiler issues all of them before a single wait (guarded loads become
  // branches with a wait each).
  for (int j0 = 0; wave + kWaves * j0 < nsteps; j0 += kSteps) {
    double a[2][kSteps][MAXRT], bv[2][kSteps];
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      const int st = wave + kWaves * (j0 + j), p = st * 4 + kq;
      const bool ok = st < nsteps;
      const bool vb = ok && cok && p < P2;
      const int pb = vb ? p : 0, pa = ok ? p : 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const double x = four[geo.at(pb, m, q, csafe)];
        bv[q][j] = vb ? x : 0.0;
#pragma unroll
        for (int r = 0; r < MAXRT; ++r)
          a[q][j][r] = W[((size_t)q * P2p + pa) * KR + (r < nrt ? r : 0) * 16];
      }
    }
#pragma unroll
    for (int j = 0; j < kSteps; ++j)
      if (wave + kWaves * (j0 + j) < nsteps)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int r = 0; r < MAXRT; ++r)
            if (r < nrt) acc[q][r] = mfma_f64(a[q][j][r], bv[q][j], acc[q][r]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int r = 0; r < MAXRT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((wave * MAXRT + r) * 4 + i) * 64 + lane] = acc[q][r][i];
    __syncthreads();
    for (int e = threadIdx.x; e < nrt * 256; e += 256) {
      const double v = red[e] + red[e + MAXRT * 256] + red[e + 2 * MAXRT * 256] + red[e + 3 * MAXRT * 256];
      const int ln = e & 63, ri = e >> 6, i = ri & 3, r = ri >> 2;
      const int k = r * 16 + i * 4 + (ln >> 4), c = ct * 16 + (ln & 15);
      if (k < kcnt[q] && c < ncol) put_spec(sm + (size_t)(2 * k + q) * ncol + c, v);
    }
    __syncthreads();
  }
}

// Wave-tile shape: one wavefront owns one 16 x 16 output tile for both parities
// and runs the whole K loop itself, so there is no cross-wave reduction, no
// LDS and no barrier, and a wave retires as soon as its tile is stored.  The
// K loop is software-pipelined over chunks of D steps (4 K values each): the
// fragments of chunk i+1 are in flight while chunk i runs on the matrix core.
// Loads go to clamped, always-valid addresses and the B operand is masked, so
// every chunk is straight-line code and the compiler keeps a running wait count.
// Units are numbered with the column tile fastest, so the four waves of a
// workgroup share table fragments (same m and row tile) in L1.

// Inverse, unit = (m, table, row tile of 16 pairs, column tile); heaviest m first.
template <int D, bool NT>
__global__ __launch_bounds__(256) void leg_inv_f64_wave_kernel(
    const double *__restrict__ spec, double *__restrict__ four, double *__restrict__ four2,
    const double *__restrict__ Pinv, const double *__restrict__ Hinv,
    const int *__restrict__ poff, const int *__restrict__ mlist, int mlen, int N, int P2, int P2p,
    int ncol, int nct, int tab0, int ntab, FourGeom geo) {
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int rtiles = P2p >> 4;
  const int upm = rtiles * ntab * nct;  // waves per m
  int m, t;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, (upm + 3) >> 2, m, t)) return;
  const int u = t * 4 + wave;
  if (u >= upm) return;
  const int ct = u % nct;
  const int rest = u / nct;
  const int rt = rest % rtiles;
  const int tab = tab0 + rest / rtiles;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KP = (ke + 3) & ~3, nsteps = KP >> 2;
  const double *__restrict__ T = (tab ? Hinv : Pinv) + poff[m] + rt * 16 + r16;
  double *__restrict__ out = tab ? four2 : four;
  const int se = tab ? 1 : 0, so = 1 - se;
  const int col = ct * 16 + r16;
  const bool cok = col < ncol;
  const double *__restrict__ sp = spec + (size_t)coef_off(N, m) * ncol + (cok ? col : 0);

  double a[2][D][2], b[2][D][2];
  auto load = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int st = s0 + j, k = st * 4 + kq;
      const int kc = st < nsteps ? k : kq;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool vb = cok && k < (q ? ko : ke);
        a[buf][j][q] = T[(size_t)(q * KP + kc) * P2p];
        const double x = sp[(size_t)(vb ? 2 * k + q : 0) * ncol];
        b[buf][j][q] = vb ? x : 0.0;
      }
    }
  };
  d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
  auto run = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (s0 + j < nsteps) {
        acc0 = mfma_f64(a[buf][j][0], b[buf][j][0], acc0);
        acc1 = mfma_f64(a[buf][j][1], b[buf][j][1], acc1);
      }
  };
  load(0, 0);
  for (int s0 = 0; s0 < nsteps; s0 += 2 * D) {
    load(1, s0 + D);
    run(0, s0);
    if (s0 + D >= nsteps) break;
    load(0, s0 + 2 * D);
    run(1, s0 + D);
  }
  if (cok) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = rt * 16 + i * 4 + kq;
      if (p < P2) {
        double *o = out + geo.tile(m, ct * 16) + (p * geo.pair() + r16);
        put_four<NT>(o + se * geo.parity(), acc0[i]);
        put_four<NT>(o + so * geo.parity(), acc1[i]);
      }
    }
  }
}

// Forward, unit = (m, 16-degree row tile, column tile) from the plan's unit
// list (m << 8 | row tile, heaviest m first); K runs over latitude pairs.
template <int D>
__global__ __launch_bounds__(256) void leg_fwd_f64_wave_kernel(
    const double *__restrict__ four, double *__restrict__ spec, const double *__restrict__ Pfwd,
    const int *__restrict__ poff, const int *__restrict__ units, int N, int P2, int P2p, int ncol,
    int nct, int nunits, FourGeom geo) {
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int u = blockIdx.x * 4 + wave;
  if (u >= nunits) return;
  const int ct = u % nct;
  const int mk = units[u / nct];
  const int m = mk >> 8, kt = mk & 255;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KR = (ke + 15) & ~15;
  const int nsteps = P2p >> 2;
  const double *__restrict__ W = Pfwd + poff[m] + kt * 16 + r16;
  const int col = ct * 16 + r16;
  const bool cok = col < ncol;
  const int csafe = cok ? col : 0;

  double a[2][D][2], b[2][D][2];
  auto load = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int st = s0 + j, p = st * 4 + kq;
      const int pa = st < nsteps ? p : kq;
      const bool vb = cok && p < P2;
      const int pb = vb ? p : 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        a[buf][j][q] = W[(size_t)(q * P2p + pa) * KR];
        const double x = four[geo.at(pb, m, q, csafe)];
        b[buf][j][q] = vb ? x : 0.0;
      }
    }
  };
  d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
  auto run = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (s0 + j < nsteps) {
        acc0 = mfma_f64(a[buf][j][0], b[buf][j][0], acc0);
        acc1 = mfma_f64(a[buf][j][1], b[buf][j][1], acc1);
      }
  };
  load(0, 0);
  for (int s0 = 0; s0 < nsteps; s0 += 2 * D) {
    load(1, s0 + D);
    run(0, s0);
    if (s0 + D >= nsteps) break;
    load(0, s0 + 2 * D);
    run(1, s0 + D);
  }
  if (cok) {
    double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol + col;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = kt * 16 + i * 4 + kq;
      if (k < ke) put_spec(sm + (size_t)(2 * k) * ncol, acc0[i]);
      if (k < ko) put_spec(sm + (size_t)(2 * k + 1) * ncol, acc1[i]);
    }
  }
}

// Tiled shape with a per-m K split.  A wave holds RT row tiles (RT*16 latitude
// pairs) of one 16-column tile in registers, so each spectral fragment it
// loads feeds RT MFMAs per parity.  The four waves of a workgroup split the K
// loop of one column tile ks ways and cover 4/ks column tiles, with ks chosen
// per m from the K length: 4 for the heavy low wavenumbers (short dependency
// chains), 1 for the light high ones (no reduction, more columns per group).
// Workgroups are numbered m-major, heaviest first: [0, m4) use ks = 4,
// [m4, m2) ks = 2, [m2, N] ks = 1 (SHT_SHAPE_TILE: m4 = m2 = 0, no split;
// SHT_SHAPE_TILE_SPLIT: thresholds on the K length).  Partial sums of a split
// meet in LDS in FP64.
template <int RT, int D, bool NT>
__global__ __launch_bounds__(256) void leg_inv_f64_tile_kernel(
    const double *__restrict__ spec, double *__restrict__ four, double *__restrict__ four2,
    const double *__restrict__ Pinv, const double *__restrict__ Hinv,
    const int *__restrict__ poff, const double *__restrict__ zero, int N, int P2, int P2p,
    int ncol, int nct, int tab0, int ntab, KSplit kspl, const int *__restrict__ mlist, int mlen,
    FourGeom geo) {
  extern __shared__ double red[];  // [4 waves][RT][4][64], one parity at a time
  const int ngr = (P2p >> 4) / RT;  // row groups
  const int w4 = ngr * ntab * nct, w2 = ngr * ntab * ((nct + 1) >> 1), w1 = ngr * ntab * ((nct + 3) >> 2);
  int b = blockIdx.x;
  int ks, m, cpw;
  if (kspl.m2 == 0) {  // no split: whole m per XCD from the balanced lists
    ks = 1; cpw = 4;
    if (!xcd_m_block(b, mlist, mlen, w1, m, b)) return;
  } else if (b < kspl.m4 * w4) {  // split regions: round robin over the XCDs
    ks = 4; cpw = 1; m = b / w4; b %= w4;
  } else if ((b -= kspl.m4 * w4) < (kspl.m2 - kspl.m4) * w2) {
    ks = 2; cpw = 2; m = kspl.m4 + b / w2; b %= w2;
  } else {
    b -= (kspl.m2 - kspl.m4) * w2;
    ks = 1; cpw = 4; m = kspl.m2 + b / w1; b %= w1;
  }
  const int ncg = (nct + cpw - 1) / cpw;
  const int ctg = b % ncg;
  b /= ncg;
  const int tab = tab0 + b % ntab;
  const int rg = b / ntab;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int kw = wave % ks, cw = wave / ks;
  const int ct = ctg * cpw + cw;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KP = (ke + 3) & ~3, nsteps = KP >> 2;
  const double *__restrict__ T = (tab ? Hinv : Pinv) + poff[m] + rg * RT * 16 + r16;
  double *__restrict__ out = tab ? four2 : four;
  const int se = tab ? 1 : 0, so = 1 - se;
  const int col = ct * 16 + r16;
  const bool cok = ct < nct && col < ncol;
  const double *__restrict__ sp = spec + (size_t)coef_off(N, m) * ncol + (cok ? col : 0);

  d4 acc[2][RT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[q][r] = d4{0.0, 0.0, 0.0, 0.0};
  // This wave's K steps are kw, kw + ks, ... < nsteps, taken in chunks of D
  // whose loads are all issued before the chunk's first MFMA.  Steps past the
  // end load clamped addresses with a zero B operand, so every MFMA is
  // unconditional (adding exact zeros) and no load can sink below a branch.
  double a[1][D][2][RT], bv[1][D][2];
  auto load = [&](int buf, int j0) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int st = kw + ks * (j0 + j), k = st * 4 + kq;
      const int kc = st < nsteps ? k : kq;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool vb = cok && k < (q ? ko : ke);
        bv[buf][j][q] = *(vb ? sp + (size_t)(2 * k + q) * ncol : zero);
#pragma unroll
        for (int r = 0; r < RT; ++r) a[buf][j][q][r] = T[(size_t)(q * KP + kc) * P2p + r * 16];
      }
    }
  };
  auto run = [&](int buf) {
#pragma unroll
    for (int j = 0; j < D; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < RT; ++r) acc[q][r] = mfma_f64(a[buf][j][q][r], bv[buf][j][q], acc[q][r]);
  };
  for (int j0 = 0; kw + ks * j0 < nsteps; j0 += D) {
    load(0, j0);
    run(0);
  }
  if (ks == 1) {
    if (cok) {
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = (rg * RT + r) * 16 + i * 4 + kq;
          if (p < P2) {
            put_four<NT>(out + geo.at(p, m, se, col), acc[0][r][i]);
            put_four<NT>(out + geo.at(p, m, so, col), acc[1][r][i]);
          }
        }
    }
    return;
  }
  // ks = 2 or 4 (uniform over the workgroup): FP64 sums of the ks partials
  const int per = RT * 256;  // doubles one wave holds per parity
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave * per + (r * 4 + i) * 64 + lane] = acc[q][r][i];
    __syncthreads();
    const int slot = q ? so : se;
    for (int e = threadIdx.x; e < cpw * per; e += 256) {
      const int g = e / per, el = e % per;
      double v = red[(g * ks) * per + el];
      for (int t = 1; t < ks; ++t) v += red[(g * ks + t) * per + el];
      const int ln = el & 63, ri = el >> 6, i = ri & 3, r = ri >> 2;
      const int p = (rg * RT + r) * 16 + i * 4 + (ln >> 4);
      const int c = (ctg * cpw + g) * 16 + (ln & 15);
      if (p < P2 && c < ncol) put_four<NT>(out + geo.at(p, m, slot, c), v);
    }
    __syncthreads();
  }
}

// Splits from the per-m K length: ks = 4 where nsteps(m) >= t4, 2 where >= t2.
inline KSplit ksplit_inv(const Plan &p, int t4, int t2) {
  KSplit k{0, 0};
  for (int m = 0; m <= p.N; ++m) {
    const int nsteps = roundup(ceil_half(p.N - m + 1), 4) / 4;
    if (nsteps >= t4) k.m4 = m + 1;
    if (nsteps >= t2) k.m2 = m + 1;
  }
  if (k.m2 < k.m4) k.m2 = k.m4;
  return k;
}

template <int RT, int D>
int inv_tile_launch(const Plan &p, KSplit ks, const double *spec, double *four, double *four2,
                    int tab0, int ntab, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const int ngr = (p.P2p / 16) / RT;
  const long w4 = (long)ngr * ntab * nct, w2 = (long)ngr * ntab * ((nct + 1) / 2),
             w1 = (long)ngr * ntab * ((nct + 3) / 4);
  const long nblk = ks.m2 == 0 ? xcd_m_blocks(p, 0, (int)w1)
                               : ks.m4 * w4 + (long)(ks.m2 - ks.m4) * w2 + (long)(p.N + 1 - ks.m2) * w1;
  const size_t lds = ks.m2 > 0 ? sizeof(double) * 4 * RT * 256 : 0;
  const FourGeom geo = four_geom_out(p, nf, sizeof(double));
  launch_kernel(geo.stream ? leg_inv_f64_tile_kernel<RT, D, true> : leg_inv_f64_tile_kernel<RT, D, false>,
      (int)nblk, 256, lds, s, spec, four, four2, p.Pinv, p.Hinv, p.poff_inv, p.zero, p.N, p.P2,
      p.P2p, ncol, nct, tab0, ntab, ks, p.xcd_m[0], p.xcd_mlen[0], geo);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

template <int D>
int inv_wave_launch(const Plan &p, const double *spec, double *four, double *four2, int tab0,
                    int ntab, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const int upm = ntab * (p.P2p / 16) * nct;
  const FourGeom geo = four_geom_out(p, nf, sizeof(double));
  launch_kernel(geo.stream ? leg_inv_f64_wave_kernel<D, true> : leg_inv_f64_wave_kernel<D, false>,
      xcd_m_blocks(p, 0, (upm + 3) / 4), 256, 0, s, spec, four, four2, p.Pinv, p.Hinv, p.poff_inv,
      p.xcd_m[0], p.xcd_mlen[0], p.N, p.P2, p.P2p, ncol, nct, tab0, ntab, geo);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

// Forward counterpart: a wave holds all 16-degree row tiles of its m (at most
// MAXRT) for one column tile, so each Fourier fragment feeds every row tile;
// the latitude-pair loop is split ks ways per m as in the inverse, with ks
// chosen from the number of row tiles (the work of an m).
template <int MAXRT, int D>
__global__ __launch_bounds__(256) void leg_fwd_f64_tile_kernel(
    const double *__restrict__ four, double *__restrict__ spec, const double *__restrict__ Pfwd,
    const int *__restrict__ poff, const double *__restrict__ zero, int N, int P2, int P2p,
    int ncol, int nct, KSplit kspl, const int *__restrict__ mlist, int mlen, FourGeom geo) {
  extern __shared__ double red[];  // [4 waves][MAXRT][4][64], one parity at a time
  const int w4 = nct, w2 = (nct + 1) >> 1, w1 = (nct + 3) >> 2;
  int b = blockIdx.x;
  int ks, m, cpw;
  if (kspl.m2 == 0) {  // no split: whole m per XCD from the balanced lists
    ks = 1; cpw = 4;
    if (!xcd_m_block(b, mlist, mlen, w1, m, b)) return;
  } else if (b < kspl.m4 * w4) {  // split regions: round robin over the XCDs
    ks = 4; cpw = 1; m = b / w4; b %= w4;
  } else if ((b -= kspl.m4 * w4) < (kspl.m2 - kspl.m4) * w2) {
    ks = 2; cpw = 2; m = kspl.m4 + b / w2; b %= w2;
  } else {
    b -= (kspl.m2 - kspl.m4) * w2;
    ks = 1; cpw = 4; m = kspl.m2 + b / w1; b %= w1;
  }
  const int ctg = b;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int kw = wave % ks, cw = wave / ks;
  const int ct = ctg * cpw + cw;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KR = (ke + 15) & ~15, nrt = KR >> 4;
  const int nsteps = P2p >> 2;
  const double *__restrict__ W = Pfwd + poff[m] + r16;
  const int col = ct * 16 + r16;
  const bool cok = ct < nct && col < ncol;
  const int csafe = cok ? col : 0;

  d4 acc[2][MAXRT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < MAXRT; ++r) acc[q][r] = d4{0.0, 0.0, 0.0, 0.0};
  // Chunks of D latitude-pair steps as in the inverse.  Row tiles past this
  // m's last (r >= nrt) reuse tile 0's fragment and their results are never
  // stored: unconditional MFMAs keep every load early.
  double a[1][D][2][MAXRT], bv[1][D][2];
  auto load = [&](int buf, int j0) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int st = kw + ks * (j0 + j), p = st * 4 + kq;
      const int pa = st < nsteps ? p : kq;
      const bool vb = cok && p < P2;
      const int pb = vb ? p : 0;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        bv[buf][j][q] = *(vb ? four + geo.at(pb, m, q, csafe) : zero);
#pragma unroll
        for (int r = 0; r < MAXRT; ++r)
          a[buf][j][q][r] = W[(size_t)(q * P2p + pa) * KR + (r < nrt ? r : 0) * 16];
      }
    }
  };
  auto run = [&](int buf) {
#pragma unroll
    for (int j = 0; j < D; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < MAXRT; ++r) acc[q][r] = mfma_f64(a[buf][j][q][r], bv[buf][j][q], acc[q][r]);
  };
  for (int j0 = 0; kw + ks * j0 < nsteps; j0 += D) {
    load(0, j0);
    run(0);
  }
  double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol;
  const int kcnt[2] = {ke, ko};
  if (ks == 1) {
    if (cok) {
#pragma unroll
      for (int r = 0; r < MAXRT; ++r)
        if (r < nrt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = r * 16 + i * 4 + kq;
            if (k < ke) put_spec(sm + (size_t)(2 * k) * ncol + col, acc[0][r][i]);
            if (k < ko) put_spec(sm + (size_t)(2 * k + 1) * ncol + col, acc[1][r][i]);
          }
    }
    return;
  }
  const int per = nrt * 256;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int r = 0; r < MAXRT; ++r)
      if (r < nrt)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave * per + (r * 4 + i) * 64 + lane] = acc[q][r][i];
    __syncthreads();
    for (int e = threadIdx.x; e < cpw * per; e += 256) {
      const int g = e / per, el = e % per;
      double v = red[(g * ks) * per + el];
      for (int t = 1; t < ks; ++t) v += red[(g * ks + t) * per + el];
      const int ln = el & 63, ri = el >> 6, i = ri & 3, r = ri >> 2;
      const int k = r * 16 + i * 4 + (ln >> 4);
      const int c = (ctg * cpw + g) * 16 + (ln & 15);
      if (k < kcnt[q] && c < ncol) put_spec(sm + (size_t)(2 * k + q) * ncol + c, v);
    }
    __syncthreads();
  }
}

// ks = 4 where the m has at least t4 row tiles, 2 where at least t2.
inline KSplit ksplit_fwd(const Plan &p, int t4, int t2) {
  KSplit k{0, 0};
  for (int m = 0; m <= p.N; ++m) {
    const int nrt = roundup(ceil_half(p.N - m + 1), 16) / 16;
    if (nrt >= t4) k.m4 = m + 1;
    if (nrt >= t2) k.m2 = m + 1;
  }
  if (k.m2 < k.m4) k.m2 = k.m4;
  return k;
}

template <int MAXRT, int D>
int fwd_tile_launch(const Plan &p, KSplit ks, const double *four, double *spec, int nf,
                    hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const long nblk = ks.m2 == 0 ? xcd_m_blocks(p, 1, (nct + 3) / 4)
                               : (long)ks.m4 * nct + (long)(ks.m2 - ks.m4) * ((nct + 1) / 2) +
                                     (long)(p.N + 1 - ks.m2) * ((nct + 3) / 4);
  const size_t lds = ks.m2 > 0 ? sizeof(double) * 4 * MAXRT * 256 : 0;
  launch_kernel(leg_fwd_f64_tile_kernel<MAXRT, D>, (int)nblk, 256, lds, s,
      four, spec, p.Pfwd, p.poff_fwd, p.zero, p.N, p.P2, p.P2p, ncol, nct, ks, p.xcd_m[1],
      p.xcd_mlen[1], four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

template <int D>
int fwd_wave_launch(const Plan &p, const double *four, double *spec, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const int nunits = p.n_fwd_units * nct;
  launch_kernel(leg_fwd_f64_wave_kernel<D>, (nunits + 3) / 4, 256, 0, s,
      four, spec, p.Pfwd, p.poff_fwd, p.fwd_units, p.N, p.P2, p.P2p, ncol, nct, nunits,
      four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

// Staged shape: the workgroup copies the data block of its (m, CT column
// tiles) into LDS once -- for the forward all latitude pairs and both
// parities of the Fourier data, for the inverse all degrees of the spectra --
// and wave w then takes the (parity, 16-row tile) units w, w+NW, ... and runs
// each over the whole K loop: table fragments from global memory (one per
// step, used for all CT column tiles), data fragments from LDS.  No partial
// sums cross waves, and a wave holds only CT accumulators and its table
// pipeline, so occupancy is set by the LDS block alone.  Built for the large
// truncations, where the other shapes re-read the data tile per row tile or
// hold every row tile's accumulators at once.  Per output tile the MFMA
// sequence depends neither on NW nor on CT.
//
// NW waves share the block: from P2p = 128 latitude pairs (the T170 grid)
// eight, and the inverse there takes two column tiles (each table fragment
// feeds two MFMAs, halving the table traffic from L2) except in small calls
// (kOneTileMaxFields); below that four waves and one column tile.  Measured at T170, 776 fields: inverse 248 against
// 273 us with four waves and one tile, forward 277 against 295 us (two tiles
// for the forward: 276 us, but slower at 97 and 388 fields); eight waves were
// slower at T42 and T85.  Measured no faster: table loads 8 or 16 steps
// ahead instead of 4, two accumulator chains per unit, staging rows
// parity-fastest or in one round of loads; slower: holding a wave's results
// until its last unit with a chunk's LDS data read ahead (T170 forward 320
// against 296 us).
//
// Copies rows of 16 columns of CT column tiles with NT threads: element e of a
// tile's block is the column pair c2 = e % 8 of row r = e / 8; src(j, r, col)
// returns columns col, col + 1 (col even) of the row in tile j (a constant, so
// tile bases stay scalar), zeros outside the data.  NQ loads per tile are
// issued before their LDS stores.
template <int NQ, int NT, int CT, class Src>
__device__ __forceinline__ void stage_rows(double *sb, int nrow, Src src) {
  const int nel = nrow * 8;
  for (int e0 = threadIdx.x; e0 < nel; e0 += NQ * NT) {
    double2 v[CT][NQ];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int e = e0 + q * NT;
        v[j][q] = e < nel ? src(j, e >> 3, 2 * (e & 7)) : make_double2(0.0, 0.0);
      }
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int e = e0 + q * NT;
        if (e < nel) *reinterpret_cast<double2 *>(sb + 2 * (j * nel + e)) = v[j][q];
      }
  }
}
// A unit's table rows: the lane's value of step s (4 K values) lies `lane`
// bytes into row group w + s * pitch.  w is the same in all lanes, so a load
// is a scalar base and one constant lane offset.
struct TableCol {
  const double *w;
  unsigned lane, pitch;
  int nsteps;
};

// One unit: acc[c] += A(s) B_c(s) over the table's steps in order; b points at
// the lane's value of step 0 of column tile 0 in LDS (64 doubles a step,
// `tile` doubles a column tile).  Table values (global memory) and data run a
// chunk of D steps ahead of the matrix core in straight-line code: with a
// branch per step every MFMA waited for its own LDS read (about 240 cycles a
// step, of which 64 are the MFMA's).  T85, 97 fields: inverse 9.4 -> 8.1 us,
// forward 9.7 -> 9.4; T170, 145 fields: 50.9 -> 47.4 and 52.6 -> 49.2; 776
// fields: 214 -> 211 and 248 -> 227.  On entry a[0] holds the table's first
// chunk (chunk(0, cur, 0)), on return the first chunk of `next`, the wave's
// next unit.  The steps that fill up the last chunk are loaded and not run: up
// to kStepSlack steps past the unit's table (still inside the plan's, which is
// that much longer) and past its data in LDS.
template <int CT, int D>
struct StagedUnit {
  static_assert(D - 1 <= kStepSlack, "slack");
  double a[2][D];
  __device__ __forceinline__ void chunk(int buf, const TableCol &t, int c) {
    const double *w = t.w + (size_t)c * D * t.pitch;
#pragma unroll
    for (int j = 0; j < D; ++j)
      a[buf][j] = *reinterpret_cast<const double *>(reinterpret_cast<const char *>(w + (size_t)j * t.pitch) + t.lane);
  }
  __device__ __forceinline__ void run(const TableCol &cur, const TableCol &next, const double *b, int tile,
                                      d4 (&acc)[CT]) {
    // data one chunk ahead where the registers allow it
    constexpr int NB = CT > 1 ? 1 : 2;
    double x[NB][CT][D];
    auto read = [&](int buf, int c) {
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int j = 0; j < D; ++j) x[buf % NB][i][j] = b[i * tile + (c * D + j) * 64];
    };
    auto mma = [&](int buf, int n) {
#pragma unroll
      for (int j = 0; j < D; ++j) {
        if (j >= n) break;
#pragma unroll
        for (int i = 0; i < CT; ++i) acc[i] = mfma_f64(a[buf][j], x[buf % NB][i][j], acc[i]);
      }
    };
    auto ahead = [&](int buf, int c) { if constexpr (NB == 2) read(buf, c); };
    auto now = [&](int c) { if constexpr (NB == 1) read(0, c); };
    const int nfull = cur.nsteps / D, rem = cur.nsteps - nfull * D, last = rem ? nfull : nfull - 1;
    ahead(0, 0);
    int c = 0;
    for (; c + 2 <= nfull; c += 2) {
      chunk(1, cur, c + 1);
      ahead(1, c + 1);
      now(c);
      mma(0, D);
      const bool more = c + 2 <= last;
      chunk(0, more ? cur : next, more ? c + 2 : 0);
      ahead(0, more ? c + 2 : last);
      now(c + 1);
      mma(1, D);
    }
    if (c < nfull) {
      chunk(1, cur, last);
      ahead(1, last);
      now(c);
      mma(0, D);
      chunk(0, next, 0);
      now(last);
      mma(1, rem);
    } else if (rem) {
      now(c);
      mma(0, rem);
      chunk(0, next, 0);
    }
  }
};

// Forward, workgroup = (m, CT column tiles); LDS [CT][parity][P2p pairs][16].
template <int CT, int D, int NW>
__device__ __forceinline__ void leg_fwd_f64_staged_item(
    double *sb, const double *__restrict__ four, double *__restrict__ spec, const double *__restrict__ Pfwd,
    const int *__restrict__ poff, int N, int P2, int P2p, int ncol, FourGeom geo, int m, int t) {
  const int ct0 = t * CT;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KR = (ke + 15) & ~15, nrt = KR >> 4;
  auto table = [&](int u) {  // units past the last: unit 0, loaded but not run
    const int uc = u < 2 * nrt ? u : 0, q = uc & 1, rt = uc >> 1;
    return TableCol{Pfwd + poff[m] + (size_t)q * P2p * KR + rt * 16, (kq * KR + r16) * 8u, 4u * KR, P2p >> 2};
  };
  StagedUnit<CT, D> unit;
  unit.chunk(0, table(wave), 0);
  // the Fourier scratch is 16-byte aligned and its column runs are even
  stage_rows<4, NW * 64, CT>(sb, 2 * P2p, [&](int j, int r, int c) {
    const int par = r >= P2p, p = r - par * P2p, col = (ct0 + j) * 16;
    return (p < P2 && col + c < ncol) ? *reinterpret_cast<const double2 *>(
                                            four + geo.tile(m, col) + (p * geo.pair() + par * geo.parity() + c))
                                      : make_double2(0.0, 0.0);
  });
  __syncthreads();
  double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol;
  for (int u = wave; u < 2 * nrt; u += NW) {
    const int q = u & 1, rt = u >> 1;
    const double *B = sb + (q * P2p + kq) * 16 + r16;
    d4 acc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] = d4{0.0, 0.0, 0.0, 0.0};
    unit.run(table(u), table(u + NW), B, 2 * P2p * 16, acc);
    const int kn = q ? ko : ke;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = (ct0 + c) * 16 + r16;
      if (col < ncol)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = rt * 16 + i * 4 + kq;
          if (k < kn) put_spec(sm + (size_t)(2 * k + q) * ncol + col, acc[c][i]);
        }
    }
  }
}

template <int CT, int D, int NW>
__global__ __launch_bounds__(NW * 64) void leg_fwd_f64_staged_kernel(
    const double *__restrict__ four, double *__restrict__ spec, const double *__restrict__ Pfwd,
    const int *__restrict__ poff, const int *__restrict__ mlist, int mlen, int N, int P2, int P2p,
    int ncol, int nct, FourGeom geo) {
  extern __shared__ double sb[];
  int m, t;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, (nct + CT - 1) / CT, m, t)) return;
  leg_fwd_f64_staged_item<CT, D, NW>(sb, four, spec, Pfwd, poff, N, P2, P2p, ncol, geo, m, t);
}

// Inverse, workgroup = (m, table or tables, CT column tiles); LDS [CT][parity][KP][16]
// with KP = this m's degrees per parity rounded up to 4 (rows past a parity's
// last degree hold zeros).
// MERGE: both tables, the value table's units first; else table tab0.
template <int CT, int D, int NW, bool NT, bool MERGE>
__device__ __forceinline__ void leg_inv_f64_staged_item(
    double *sb, const double *__restrict__ spec, double *__restrict__ four, double *__restrict__ four2,
    const double *__restrict__ Pinv, const double *__restrict__ Hinv, const int *__restrict__ poff, int N, int P2,
    int P2p, int ncol, FourGeom geo, int m, int tab0, int ct0) {
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KP = (ke + 3) & ~3;
  const double *__restrict__ sp = spec + (size_t)coef_off(N, m) * ncol;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int half = P2p >> 3, nunits = MERGE ? 2 * half : half;  // a table's units: 2 parities x 16-row tiles
  auto table = [&](int u) {  // units past the last: unit 0, loaded but not run
    const int uc = u < nunits ? u : 0, second = MERGE && uc >= half, tab = MERGE ? second : tab0, q = uc & 1,
              rt = (second ? uc - half : uc) >> 1;
    return TableCol{(tab ? Hinv : Pinv) + poff[m] + (size_t)q * KP * P2p + rt * 16, (kq * P2p + r16) * 8u, 4u * P2p,
                    KP >> 2};
  };
  StagedUnit<CT, D> unit;
  unit.chunk(0, table(wave), 0);
  // the caller's spectra may be only 8-byte aligned: two loads per pair
  stage_rows<4, NW * 64, CT>(sb, 2 * KP, [&](int j, int r, int c) {
    const int par = r >= KP, k = r - par * KP, col = (ct0 + j) * 16 + c;
    if (k >= (par ? ko : ke) || col >= ncol) return make_double2(0.0, 0.0);
    const double *x = sp + (size_t)(2 * k + par) * ncol + col;
    return make_double2(x[0], x[1]);
  });
  __syncthreads();
  for (int u = wave; u < nunits; u += NW) {
    const int second = MERGE && u >= half, tab = MERGE ? second : tab0, q = u & 1, rt = (second ? u - half : u) >> 1;
    double *__restrict__ out = tab ? four2 : four;
    const int se = tab ? 1 : 0;  // the derivative table's parities are swapped
    const double *B = sb + (q * KP + kq) * 16 + r16;
    d4 acc[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[c] = d4{0.0, 0.0, 0.0, 0.0};
    unit.run(table(u), table(u + NW), B, 2 * KP * 16, acc);
    const int slot = q ^ se;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = (ct0 + c) * 16 + r16;
      if (col < ncol)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int p = rt * 16 + i * 4 + kq;
          if (p < P2)
            put_four<NT>(out + geo.tile(m, (ct0 + c) * 16) + (p * geo.pair() + slot * geo.parity() + r16), acc[c][i]);
        }
    }
  }
}

template <int CT, int D, int NW, bool NT, bool MERGE>
__global__ __launch_bounds__(NW * 64) void leg_inv_f64_staged_kernel(
    const double *__restrict__ spec, double *__restrict__ four, double *__restrict__ four2,
    const double *__restrict__ Pinv, const double *__restrict__ Hinv, const int *__restrict__ poff,
    const int *__restrict__ mlist, int mlen, int N, int P2, int P2p, int ncol, int nct, int tab0,
    int ntab, FourGeom geo) {
  extern __shared__ double sb[];
  const int ncg = (nct + CT - 1) / CT;
  int m, t;
  const int per = MERGE ? 1 : ntab;  // workgroups per column group
  if (!xcd_m_block(blockIdx.x, mlist, mlen, per * ncg, m, t)) return;
  leg_inv_f64_staged_item<CT, D, NW, NT, MERGE>(sb, spec, four, four2, Pinv, Hinv, poff, N, P2, P2p, ncol, geo, m,
                                         tab0 + t % per, (t / per) * CT);
}

// ---- Several groups in one launch (sht_internal.h, MultiGroup): the staged
// shape with one column tile and four waves, workgroup ranges per group.
struct F64Multi {
  int ng;
  struct Group {
    const double *spec_in;
    double *four, *spec_out;
    const double *table;
    const int *poff, *mlist;
    int blk0, mlen, N, P2, P2p, ncol, nct;
    FourGeom geo;
  } g[kMaxMulti];
};

template <bool FWD, bool NT>
__global__ __launch_bounds__(256) void leg_f64_multi_kernel(F64Multi a) {
  extern __shared__ double sb[];
  const F64Multi::Group &g = a.g[multi_group(a, blockIdx.x)];
  int m, t;
  if (!xcd_m_block(blockIdx.x - g.blk0, g.mlist, g.mlen, g.nct, m, t)) return;
  if constexpr (FWD)
    leg_fwd_f64_staged_item<1, 4, 4>(sb, g.four, g.spec_out, g.table, g.poff, g.N, g.P2, g.P2p, g.ncol, g.geo, m, t);
  else
    leg_inv_f64_staged_item<1, 4, 4, NT, false>(sb, g.spec_in, g.four, nullptr, g.table, nullptr, g.poff, g.N, g.P2, g.P2p,
                                         g.ncol, g.geo, m, 0, t);
}

inline size_t fwd_staged_lds(const Plan &p, int ct) {
  return sizeof(double) * ct * 2 * p.P2p * 16;  // <= 64 KB: P2p <= 256
}
inline size_t inv_staged_lds(const Plan &p, int ct) {
  // the last tile's rows filled up to a chunk of 16; <= 64 KB: kp0 <= 128
  const int kp0 = roundup(ceil_half(p.N + 1), 4);
  return sizeof(double) * ((ct * 2 - 1) * kp0 + roundup(kp0, 16)) * 16;
}

template <int CT, int NW>
int fwd_staged_launch(const Plan &p, const double *four, double *spec, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  launch_kernel(leg_fwd_f64_staged_kernel<CT, 4, NW>, xcd_m_blocks(p, 1, (nct + CT - 1) / CT), NW * 64,
      fwd_staged_lds(p, CT), s, four, spec, p.Pfwd, p.poff_fwd, p.xcd_m[1], p.xcd_mlen[1], p.N, p.P2, p.P2p, ncol, nct,
      four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

template <int CT, int NW>
int inv_staged_launch(const Plan &p, const double *spec, double *four, double *four2, int tab0,
                      int ntab, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const FourGeom geo = four_geom_out(p, nf, sizeof(double));
  // both tables in one workgroup: the spectra are staged once, but half as many
  // workgroups run twice as long, so only where those fill the chip (2048 are two
  // rounds of four per CU), or half as many if a wave has one unit per table and
  // the staging is most of a workgroup's life.  Gradients' Legendre step, one
  // table / both per workgroup: T21 400 fields 6.6 / 6.0 us; T42 79 fields 5.8 / 5.7,
  // 192 fields 7.9 / 6.8, 388 fields 13.1 / 10.6; T85 97 fields 12.0 / 12.6, 190 fields
  // 23.8 / 22.0; T170 64 fields 40.8 / 44.9, 192 fields 111 / 107.
  const int nwg = xcd_m_blocks(p, 0, (nct + CT - 1) / CT);
  const bool merge = ntab == 2 && nwg >= (p.P2p / 8 <= NW ? 1024 : 2048);
  auto kern = geo.stream ? leg_inv_f64_staged_kernel<CT, 4, NW, true, false> : leg_inv_f64_staged_kernel<CT, 4, NW, false, false>;
  if constexpr (CT > 1 || NW < 8)  // one tile and eight waves: one table only (kOneTileMaxFields)
    if (merge) kern = geo.stream ? leg_inv_f64_staged_kernel<CT, 4, NW, true, true> : leg_inv_f64_staged_kernel<CT, 4, NW, false, true>;
  launch_kernel(kern,
      merge ? nwg : xcd_m_blocks(p, 0, ntab * ((nct + CT - 1) / CT)), NW * 64, inv_staged_lds(p, CT), s, spec, four, four2, p.Pinv, p.Hinv,
      p.poff_inv, p.xcd_m[0], p.xcd_mlen[0], p.N, p.P2, p.P2p, ncol, nct, tab0, ntab, geo);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

// Staged in two parts: the forward for larger batches on the T170 grid.  The
// latitude pairs are staged and run in two halves, so the LDS block of half of
// them holds two column tiles and each table value feeds two MFMAs.  The steps
// of an output tile still run in order from a zero accumulator, so results are
// bitwise those of the one-part kernel; a wave's MAXU units keep their
// accumulators across the halves and store after the second.  Measured at T170
// (eight waves), one part / two: 33 fields 16.1 / 16.0 us, 97 fields 36.5 / 34.4,
// 145 fields 50.2 / 46.5, 388 fields 133 / 123, 776 fields 267 / 237.  (The
// inverse, whose two-tile block fits whole, gains nothing: with four tiles 388
// fields 119 against 113 us, 776 fields 218 against 206.)
// LDS [CT][parity][P2p / 2 pairs][16].
template <int CT, int D, int NW, int MAXU>
__global__ __launch_bounds__(NW * 64) void leg_fwd_f64_halves_kernel(
    const double *__restrict__ four, double *__restrict__ spec, const double *__restrict__ Pfwd,
    const int *__restrict__ poff, const int *__restrict__ mlist, int mlen, int N, int P2, int P2p,
    int ncol, int nct, FourGeom geo) {
  extern __shared__ double sb[];
  int m, t;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, (nct + CT - 1) / CT, m, t)) return;
  const int ct0 = t * CT, H = P2p >> 1;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KR = (ke + 15) & ~15, nrt = KR >> 4;
  d4 acc[MAXU][CT];
#pragma unroll
  for (int i = 0; i < MAXU; ++i)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[i][c] = d4{0.0, 0.0, 0.0, 0.0};
  auto table = [&](int h, int u) {  // units past the last: unit 0, loaded but not run
    const int uc = u < 2 * nrt ? u : 0, q = uc & 1, rt = uc >> 1;
    return TableCol{Pfwd + poff[m] + ((size_t)q * P2p + h * H) * KR + rt * 16, (kq * KR + r16) * 8u, 4u * KR, H >> 2};
  };
  StagedUnit<CT, D> unit;
  unit.chunk(0, table(0, wave), 0);
  for (int h = 0; h < 2; ++h) {
    if (h) __syncthreads();
    stage_rows<2, NW * 64, CT>(sb, 2 * H, [&](int j, int r, int c) {
      const int par = r >= H, p = h * H + (r - par * H), col = (ct0 + j) * 16;
      return (p < P2 && col + c < ncol) ? *reinterpret_cast<const double2 *>(
                                              four + geo.tile(m, col) + (p * geo.pair() + par * geo.parity() + c))
                                        : make_double2(0.0, 0.0);
    });
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MAXU; ++i) {
      const int u = wave + NW * i, q = u & 1, un = u + NW;
      if (u >= 2 * nrt) break;
      const bool last = i + 1 == MAXU || un >= 2 * nrt;  // of this half
      const double *B = sb + (q * H + kq) * 16 + r16;
      unit.run(table(h, u), last ? table(1, wave) : table(h, un), B, 2 * H * 16, acc[i]);
    }
  }
  double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol;
#pragma unroll
  for (int i = 0; i < MAXU; ++i) {
    const int u = wave + NW * i, q = u & 1, rt = u >> 1;
    if (u >= 2 * nrt) break;
    const int kn = q ? ko : ke;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const int col = (ct0 + c) * 16 + r16;
      if (col < ncol)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = rt * 16 + j * 4 + kq;
          if (k < kn) put_spec(sm + (size_t)(2 * k + q) * ncol + col, acc[i][c][j]);
        }
    }
  }
}

// Divergence analysis: spec = Pfwd fa + Hfwd fb, either input absent (NULL).
// The H table holds (1-mu^2) dPt/dmu, of the opposite equatorial parity, so
// the parity-q degrees read slot 1 - q of fb.  The staged shape with the K
// range being the pairs of fa, then those of fb: a workgroup stages one input
// after the other and keeps its units' accumulators, so both terms leave in
// one store and the spectra are never read back.  Both inputs' loads (NQ per
// thread and input) are in flight before the first is staged.  T85, 65 fields:
// 12.0 us against 17.8 us for two K-split launches, the second adding into the
// first's output.
template <int NW, int NQ>
__global__ __launch_bounds__(NW * 64) void leg_fwd_f64_div_kernel(
    const double *__restrict__ fa, const double *__restrict__ fb, double *__restrict__ spec,
    const double *__restrict__ Pfwd, const double *__restrict__ Hfwd, const int *__restrict__ poff,
    const int *__restrict__ mlist, int mlen, int N, int P2, int P2p, int ncol, int nct, FourGeom geo) {
  constexpr int MAXU = 2;
  extern __shared__ double sb[];  // [parity][P2p pairs][16]
  int m, ct;
  if (!xcd_m_block(blockIdx.x, mlist, mlen, nct, m, ct)) return;
  const int wave = wave_id(), lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
  const int nn = N - m + 1, ke = (nn + 1) >> 1, ko = nn >> 1;
  const int KR = (ke + 15) & ~15, nrt = KR >> 4;
  d4 acc[MAXU][1];
#pragma unroll
  for (int i = 0; i < MAXU; ++i) acc[i][0] = d4{0.0, 0.0, 0.0, 0.0};
  // element e of an input's block: column pair e % 8 of (parity, pair) row e / 8
  double2 v[2][NQ];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int e = threadIdx.x + i * NW * 64, r = e >> 3, par = r >= P2p, p = r - par * P2p;
      const int c = 2 * (e & 7);
      const double *four = h ? fb : fa;
      const bool ok = four && r < 2 * P2p && p < P2 && ct * 16 + c < ncol;
      v[h][i] = ok ? *reinterpret_cast<const double2 *>(four + geo.tile(m, ct * 16) +
                                                        (p * geo.pair() + par * geo.parity() + c))
                   : make_double2(0.0, 0.0);
    }
  auto table = [&](int h, int u) {  // units past the last: unit 0, loaded but not run
    const int uc = u < 2 * nrt ? u : 0, q = uc & 1, rt = uc >> 1;
    return TableCol{(h ? Hfwd : Pfwd) + poff[m] + (size_t)q * P2p * KR + rt * 16, (kq * KR + r16) * 8u, 4u * KR,
                    P2p >> 2};
  };
  const int h0 = fa ? 0 : 1, h1 = fb ? 1 : 0;  // the inputs that are present
  StagedUnit<1, 4> unit;
  unit.chunk(0, table(h0, wave), 0);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h < h0 || h > h1) continue;
    if (h) __syncthreads();
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int e = threadIdx.x + i * NW * 64;
      if (e < 16 * P2p) *reinterpret_cast<double2 *>(sb + 2 * e) = v[h][i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MAXU; ++i) {
      const int u = wave + NW * i, q = u & 1, un = u + NW;
      if (u >= 2 * nrt) break;
      const bool last = i + 1 == MAXU || un >= 2 * nrt;  // of this input
      const double *B = sb + ((q ^ h) * P2p + kq) * 16 + r16;
      unit.run(table(h, u), last ? table(h1, wave) : table(h, un), B, 0, acc[i]);
    }
  }
  const int col = ct * 16 + r16;
  if (col >= ncol) return;
  double *__restrict__ sm = spec + (size_t)coef_off(N, m) * ncol + col;
#pragma unroll
  for (int i = 0; i < MAXU; ++i) {
    const int u = wave + NW * i, q = u & 1, rt = u >> 1;
    if (u >= 2 * nrt) break;
    const int kn = q ? ko : ke;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = rt * 16 + j * 4 + kq;
      if (k < kn) put_spec(sm + (size_t)(2 * k + q) * ncol, acc[i][0][j]);
    }
  }
}

template <int NW, int NQ>
int fwd_div_launch(const Plan &p, const double *fa, const double *fb, double *spec, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const size_t lds = sizeof(double) * 2 * p.P2p * 16;  // <= 64 KB: P2p <= 256
  launch_kernel(leg_fwd_f64_div_kernel<NW, NQ>, xcd_m_blocks(p, 1, nct), NW * 64, lds, s, fa, fb, spec, p.Pfwd,
                p.Hfwd, p.poff_fwd, p.xcd_m[1], p.xcd_mlen[1], p.N, p.P2, p.P2p, ncol, nct, four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

template <bool FWD>
int f64_multi_launch(const MultiGroup *g, int n, hipStream_t s) {
  F64Multi a{};
  a.ng = n;
  int nblk = 0;
  size_t lds = 0;
  for (int i = 0; i < n; ++i) {
    const Plan &p = *g[i].p;
    const int ncol = 2 * g[i].nf, nct = (ncol + 15) / 16;
    a.g[i] = {g[i].spec_in, p.four, g[i].spec_out, FWD ? p.Pfwd : p.Pinv, FWD ? p.poff_fwd : p.poff_inv, p.xcd_m[FWD],
              nblk, p.xcd_mlen[FWD], p.N, p.P2, p.P2p, ncol, nct, multi_geom(p, g[i].nf)};
    nblk += xcd_m_blocks(p, FWD, nct);
    const size_t need = FWD ? fwd_staged_lds(p, 1) : inv_staged_lds(p, 1);
    lds = need > lds ? need : lds;
  }
  launch_kernel(FWD ? leg_f64_multi_kernel<FWD, false>
                    : (multi_streams(g, n) ? leg_f64_multi_kernel<FWD, true> : leg_f64_multi_kernel<FWD, false>),
                nblk, 256, lds, s, a);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

// Field count up to which the staged inverse of one table takes one column tile
// per workgroup on the T170 grid.  Two tiles halve the table reads, but their
// half as many workgroups (684 for 33 to 64 fields) leave the chip's last wave
// part empty: one / two tiles, Legendre step, 32 fields 12.1 / 13.7 us, 40 fields
// 15.5 / 17.6, 56 fields 19.2 / 21.1, 57 and 64 fields equal, 80 fields 29.2 / 27.3,
// 145 fields 57.2 / 50.1.  With both tables (gradients) the workgroups are twice
// as many and two tiles win from 32 fields on (24.3 / 23.2), as they do on grids
// of more latitude pairs (N = 200, 40 fields 25.1 / 23.5).  Either way each output
// tile runs the same products in the same order: the results are the same.
constexpr int kOneTileMaxFields = 56;

// Field count from which the staged forward runs in two parts on the T170 grid.
constexpr int kHalvesMinFields = 64;

// MAXU = 2: at most 2 nrt(0) <= 16 forward units over eight waves.
template <int CT, int MAXU>
int fwd_halves_launch(const Plan &p, const double *four, double *spec, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const size_t lds = sizeof(double) * CT * 2 * (p.P2p / 2) * 16;
  launch_kernel(leg_fwd_f64_halves_kernel<CT, 4, 8, MAXU>, xcd_m_blocks(p, 1, (nct + CT - 1) / CT), 512, lds,
      s, four, spec, p.Pfwd, p.poff_fwd, p.xcd_m[1], p.xcd_mlen[1], p.N, p.P2, p.P2p, ncol, nct,
      four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}
template <int RT>
int inv_launch(const Plan &p, const double *spec, double *four, double *four2, int tab0, int ntab,
               int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const int nblk = xcd_m_blocks(p, 0, ntab * nct);
  const size_t lds = sizeof(double) * kWaves * RT * 256;
  const FourGeom geo = four_geom_out(p, nf, sizeof(double));
  launch_kernel(geo.stream ? leg_inv_f64_kernel<RT, true> : leg_inv_f64_kernel<RT, false>, nblk, 256,
                lds, s, spec, four, four2, p.Pinv, p.Hinv, p.poff_inv, p.xcd_m[0], p.xcd_mlen[0], p.N,
                p.P2, p.P2p, ncol, nct, tab0, ntab, geo);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

template <int MAXRT>
int fwd_launch(const Plan &p, const double *four, double *spec, int nf, hipStream_t s) {
  const int ncol = 2 * nf, nct = (ncol + 15) / 16;
  const int nblk = xcd_m_blocks(p, 1, nct);
  const size_t lds = sizeof(double) * kWaves * MAXRT * 256;
  launch_kernel(leg_fwd_f64_kernel<MAXRT>, nblk, 256, lds, s, four, spec, p.Pfwd,
                p.poff_fwd, p.xcd_m[1], p.xcd_mlen[1], p.N, p.P2, p.P2p, ncol, nct, four_geom(p, nf));
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

}  // namespace

KSplit default_classes(const Plan &p, int dir) {
  if (dir == 0) {
    // halve the K loop of the wavenumbers with at least 70 % of the heaviest
    // one's K steps (the waves that set the critical path); no four-way
    // split.  Measured at T85: 97 fields 10.9 us (thresholds 6/3 gave 15.4,
    // TILE 13.5); T42, 388 fields 7.2 us (9.1, TILE 12.1).
    const int nsmax = roundup(ceil_half(p.N + 1), 4) / 4;
    return ksplit_inv(p, 1 << 30, (7 * nsmax + 9) / 10);
  }
  // halve the pair loop of the wavenumbers with the most row tiles only
  // (thresholds 2/1, which split every m, were slower everywhere)
  return ksplit_fwd(p, 1 << 30, roundup(ceil_half(p.N + 1), 16) / 16);
}

KSplit resolve_classes(const Plan &p, int nf, int dir) {
  for (const Plan::ShapeEntry &e : p.shapes)
    if (e.nf == nf) {
      const int m4 = dir ? e.t.fwd_m4 : e.t.inv_m4, m2 = dir ? e.t.fwd_m2 : e.t.inv_m2;
      if (m4 >= 0 && m2 >= m4 && m2 <= p.N + 1) return KSplit{m4, m2};
      break;
    }
  return default_classes(p, dir);
}

int resolve_shape(const Plan &p, int nf, int dir) {
  // an entry for nf, unless its half for this direction is AUTO
  for (const Plan::ShapeEntry &e : p.shapes)
    if (e.nf == nf) {
      const int s = dir ? e.t.fwd : e.t.inv;
      if (s != SHT_SHAPE_AUTO) return s;
      break;
    }
  const int d = dir ? p.shape_fwd : p.shape_inv;
  if (d != SHT_SHAPE_AUTO) return d;
  // mixed forms: the shapes give bitwise equal results, so the choice is by
  // speed alone -- two column tiles per workgroup from 128 latitude pairs
  // (T170: faster in both directions at 97 to 776 fields), one below.  On
  // the 128-pair grid the inverse streams (STAGED): always in the
  // six-product form, up to 8 fields and from 192 in the two-piece forms, which
  // run KSPLIT from 9 to 24 fields.  T170 inverse Legendre step, KSPLIT / TILE /
  // STAGED, us: x6 8 fields 9.4 / 9.3 / 7.2, 33 fields 15.9 / 14.0 / 13.6, 97
  // fields 31.8 / 29.6 / 25.6, 388 fields 121 / 105 / 86, 776 fields 227 / 197 /
  // 156; BF16 x3 8 fields 7.5 / 7.6 / 5.5, 17 fields 8.9 / 10.0 / 9.5, 97 fields
  // 24.3 / 21.8 / 22.1, 250 fields 66 / 56 / 52, 776 fields 177 / 146 / 140;
  // scaled FP16 97 fields 25.7 / 22.8 / 23.8, 250 fields 70 / 56 / 55, 776
  // fields 189 / 152 / 145.  Below 128 pairs the idle table waves cost more
  // than the stream saves (BF16 x3, 100 pairs, 145 fields: 17.3 / 17.7 / 18.0).
  if (p.prec != SHT_PREC_FP64) {
    if (dir == 0 && p.P2p == 128 && mixed_stream_available(p)) {
      if (p.prec == SHT_PREC_SPLIT_BF16X6 || nf <= 8 || nf >= 192) return SHT_SHAPE_STAGED;
      if (nf <= 24) return SHT_SHAPE_KSPLIT;
    }
    return p.P2p >= 128 ? SHT_SHAPE_TILE : SHT_SHAPE_KSPLIT;
  }
  // measured on MI355X from T21 to T170 and 16 to 388 fields: the staged
  // shape wins the forward nearly everywhere and the inverse from 32 fields;
  // below that a wavefront per tile fills the chip better.  STAGED, WAVE and TILE
  // run the same MFMA sequence per output tile, so the switches with the field
  // count change no result.
  // On at most 32 latitudes (up to 64 with more fields) a staged workgroup's
  // few K steps are mostly its staging, and TILE runs many fields faster, with the
  // same sequence again: STAGED / TILE, inverse, forward and both tables, us:
  // T21 (32 latitudes) 256 fields equal, equal, 5.6 / 4.8; 776 fields 6.2 / 5.6, 5.8 / 4.3,
  // 9.7 / 9.6; T10 (16 latitudes) 3000 fields 10.5 / 5.5, 11.3 / 5.4, 12.9 / 9.1; N = 31, 64
  // latitudes 388 fields 7.3 / 7.8, 5.5 / 5.3, 13.5 / 14.4; 776 fields 14.5 / 14.2, 8.9 / 7.5,
  // 18.3 / 16.2.
  if (p.P2p <= 32 && nf >= (p.P2p == 16 ? 256 : 512)) return SHT_SHAPE_TILE;
  if (dir == 1) return SHT_SHAPE_STAGED;
  return nf >= 32 ? SHT_SHAPE_STAGED : SHT_SHAPE_WAVE;
}

int launch_leg_inv_f64_shape(const Plan &p, int shape, const double *spec, double *four,
                             double *four2, bool value_table, bool deriv_table, int nf,
                             hipStream_t s, KSplit cls) {
  if (!value_table && !deriv_table) return SHT_OK;
  const int tab0 = value_table ? 0 : 1;
  const int ntab = (value_table && deriv_table) ? 2 : 1;
  if (shape == SHT_SHAPE_WAVE) return inv_wave_launch<4>(p, spec, four, four2, tab0, ntab, nf, s);
  if (shape == SHT_SHAPE_STAGED) {
    if (p.P2p < 128) return inv_staged_launch<1, 4>(p, spec, four, four2, tab0, ntab, nf, s);
    if (p.P2p == 128 && ntab == 1 && nf <= kOneTileMaxFields)
      return inv_staged_launch<1, 8>(p, spec, four, four2, tab0, ntab, nf, s);
    return inv_staged_launch<2, 8>(p, spec, four, four2, tab0, ntab, nf, s);
  }
  if (shape == SHT_SHAPE_TILE || shape == SHT_SHAPE_TILE_SPLIT) {
    const int rtiles = p.P2p / 16;
    int rt = 4;
    while (rtiles % rt) --rt;
    // TILE_SPLIT: the given wavenumber classes, else the built-in ones
    const KSplit k = shape == SHT_SHAPE_TILE ? KSplit{0, 0} : (cls.m2 >= 0 ? cls : default_classes(p, 0));
    switch (rt) {
      case 4: return inv_tile_launch<4, 2>(p, k, spec, four, four2, tab0, ntab, nf, s);
      case 3: return inv_tile_launch<3, 2>(p, k, spec, four, four2, tab0, ntab, nf, s);
      case 2: return inv_tile_launch<2, 2>(p, k, spec, four, four2, tab0, ntab, nf, s);
      default: return inv_tile_launch<1, 2>(p, k, spec, four, four2, tab0, ntab, nf, s);
    }
  }
  const int rtiles = p.P2p / 16;
  int rt = 8;
  while (rtiles % rt) --rt;
  switch (rt) {
    case 8: return inv_launch<8>(p, spec, four, four2, tab0, ntab, nf, s);
    case 7: return inv_launch<7>(p, spec, four, four2, tab0, ntab, nf, s);
    case 6: return inv_launch<6>(p, spec, four, four2, tab0, ntab, nf, s);
    case 5: return inv_launch<5>(p, spec, four, four2, tab0, ntab, nf, s);
    case 4: return inv_launch<4>(p, spec, four, four2, tab0, ntab, nf, s);
    case 3: return inv_launch<3>(p, spec, four, four2, tab0, ntab, nf, s);
    case 2: return inv_launch<2>(p, spec, four, four2, tab0, ntab, nf, s);
    default: return inv_launch<1>(p, spec, four, four2, tab0, ntab, nf, s);
  }
}

int launch_leg_fwd_f64_shape(const Plan &p, int shape, const double *four, double *spec, int nf,
                             hipStream_t s, KSplit cls) {
  if (shape == SHT_SHAPE_WAVE) return fwd_wave_launch<4>(p, four, spec, nf, s);
  if (shape == SHT_SHAPE_STAGED && p.P2p == 128 && nf >= kHalvesMinFields)
    return fwd_halves_launch<2, 2>(p, four, spec, nf, s);
  if (shape == SHT_SHAPE_STAGED)
    return p.P2p >= 128 ? fwd_staged_launch<1, 8>(p, four, spec, nf, s) : fwd_staged_launch<1, 4>(p, four, spec, nf, s);
  const int rt = (ceil_half(p.N + 1) + 15) / 16;
  if (shape == SHT_SHAPE_TILE || shape == SHT_SHAPE_TILE_SPLIT) {
    // TILE_SPLIT: the given wavenumber classes, else the built-in ones
    const KSplit k = shape == SHT_SHAPE_TILE ? KSplit{0, 0} : (cls.m2 >= 0 ? cls : default_classes(p, 1));
    switch (rt) {
      case 1: return fwd_tile_launch<1, 2>(p, k, four, spec, nf, s);
      case 2: return fwd_tile_launch<2, 2>(p, k, four, spec, nf, s);
      case 3: return fwd_tile_launch<3, 2>(p, k, four, spec, nf, s);
      case 4: return fwd_tile_launch<4, 2>(p, k, four, spec, nf, s);
      case 5: return fwd_tile_launch<5, 2>(p, k, four, spec, nf, s);
      case 6: return fwd_tile_launch<6, 2>(p, k, four, spec, nf, s);
      case 7: return fwd_tile_launch<7, 2>(p, k, four, spec, nf, s);
      case 8: return fwd_tile_launch<8, 2>(p, k, four, spec, nf, s);
    }
    return fail(SHT_ERR_UNSUPPORTED, "nmax above 255 is not instantiated");
  }
  switch (rt) {
    case 1: return fwd_launch<1>(p, four, spec, nf, s);
    case 2: return fwd_launch<2>(p, four, spec, nf, s);
    case 3: return fwd_launch<3>(p, four, spec, nf, s);
    case 4: return fwd_launch<4>(p, four, spec, nf, s);
    case 5: return fwd_launch<5>(p, four, spec, nf, s);
    case 6: return fwd_launch<6>(p, four, spec, nf, s);
    case 7: return fwd_launch<7>(p, four, spec, nf, s);
    case 8: return fwd_launch<8>(p, four, spec, nf, s);
  }
  return fail(SHT_ERR_UNSUPPORTED, "nmax above 255 is not instantiated");
}

int launch_leg_fwd_f64_div(const Plan &p, const double *fa, const double *fb, double *spec, int nf,
                           hipStream_t s) {
  // units of one m over the waves, at most two each: 2 nrt(0) <= 16
  const int units = 2 * ((ceil_half(p.N + 1) + 15) / 16);
  if (p.P2p >= 128 || units > 8)  // 16 P2p <= 4096 column pairs a block, 512 threads
    return p.P2p <= 128 ? fwd_div_launch<8, 4>(p, fa, fb, spec, nf, s) : fwd_div_launch<8, 8>(p, fa, fb, spec, nf, s);
  return p.P2p <= 64 ? fwd_div_launch<4, 4>(p, fa, fb, spec, nf, s) : fwd_div_launch<4, 7>(p, fa, fb, spec, nf, s);
}

int launch_leg_inv_f64_multi(const MultiGroup *g, int n, hipStream_t s) { return f64_multi_launch<false>(g, n, s); }
int launch_leg_fwd_f64_multi(const MultiGroup *g, int n, hipStream_t s) { return f64_multi_launch<true>(g, n, s); }

// FP64: a group takes part where its shapes run the staged shape's MFMA
// sequence (WAVE, TILE and STAGED); the mixed forms' shapes all agree.
bool multi_available(const Plan &p, int nf) {
  if (p.P2p > 64 || p.im > 256) return false;
  if (p.prec != SHT_PREC_FP64) return true;
  auto same = [](int s) { return s == SHT_SHAPE_WAVE || s == SHT_SHAPE_TILE || s == SHT_SHAPE_STAGED; };
  return same(resolve_shape(p, nf, 0)) && same(resolve_shape(p, nf, 1));
}

long multi_blocks(const Plan &p, int nf) {
  const long nct = (2L * nf + 15) / 16, gf = fft_group(p.im);
  const long leg = 8L * std::max(p.xcd_mlen[0], p.xcd_mlen[1]) * nct;
  const long fft = (long)p.P2 * multi_geom(p, nf).nfg * (layout_group(gf) / gf);
  return (std::max(leg, fft) + 7) / 8 * 8;
}

int launch_leg_inv_f64(const Plan &p, const double *spec, double *four, double *four2,
                       bool value_table, bool deriv_table, int nf, hipStream_t s) {
  return launch_leg_inv_f64_shape(p, resolve_shape(p, nf, 0), spec, four, four2, value_table,
                                  deriv_table, nf, s, resolve_classes(p, nf, 0));
}

int launch_leg_fwd_f64(const Plan &p, const double *four, double *spec, int nf, hipStream_t s) {
  return launch_leg_fwd_f64_shape(p, resolve_shape(p, nf, 1), four, spec, nf, s, resolve_classes(p, nf, 1));
}

}  // namespace sht
