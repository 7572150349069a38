// sht_remap.hip -- the coupler's grid remap on the GPU: the sparse
// interpolation of common/interpolation_data_latlon_mod.f90:274-306
// (interpolate_data_latlon), which Jcup applies to every exchanged field:
//   recv(:, d) = 0;  recv(r_i, d) += send(s_i, d) * coef_i,  i = 1..nnz
// for d = 1..ndata, fields contiguous per point (Fortran send_data(:, d)).
//
// The triplets are regrouped at creation by receiving point (CSR), keeping
// the original order within each row, and one thread sums each (row, field)
// with separately rounded multiply and add in that order: the same operations
// in the same order as the reference loop, so results are bitwise equal to an
// unfused evaluation of it (no atomics, no fused multiply-add).
#include <algorithm>
#include <new>
#include <numeric>

#include "sht_internal.h"

struct sht_remap {
  int nsend = 0, nrecv = 0, nnz = 0;
  int *row = nullptr;     // nrecv + 1 offsets
  int *col = nullptr;     // nnz send points, row-major
  double *val = nullptr;  // nnz coefficients
};

namespace sht {
namespace {

// One thread sums one row for ND fields (the last group of a call has fewer):
// row offsets, columns and coefficients are loaded once for the group, and
// kRemapAhead entries' columns, then their ND gathers each, are in flight at a
// time, where one load at a time is a chain row -> column -> value per entry.
// 32,768 rows of 4 entries, back to back: 12 fields 5.2 -> 3.9 us, 40 fields
// 13.4 -> 7.5 us; 131,072 rows, 40 fields 45.4 -> 22.6 us.  Small calls run
// single fields (ND = 1): 8,192 rows, 12 fields 3.1 -> 2.9 us.
constexpr int kRemapAhead = 4;
template <int ND>
__global__ __launch_bounds__(256) void remap_kernel(const int *__restrict__ row,
                                                    const int *__restrict__ col,
                                                    const double *__restrict__ val,
                                                    const double *__restrict__ send,
                                                    double *__restrict__ recv, int nsend, int nrecv,
                                                    int ndata) {
  // separately rounded multiply and add: hipcc otherwise contracts the pair
  // into one fused multiply-add (the operations must be written here, in the
  // pragma's scope: __dmul_rn/__dadd_rn are contracted at their definition)
#pragma clang fp contract(off)
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t total = (int64_t)nrecv * ((ndata + ND - 1) / ND);
  if (t >= total) return;
  // 32-bit division where it suffices
  const int g = total <= UINT32_MAX ? (int)((uint32_t)t / (uint32_t)nrecv) : (int)(t / nrecv);
  const int r = (int)(t - (int64_t)g * nrecv), d0 = g * ND;
  const int nd = ndata - d0 < ND ? ndata - d0 : ND;
  const double *__restrict__ s = send + (size_t)d0 * nsend;
  double acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = 0.0;
  const int end = row[r + 1];
  for (int i0 = row[r]; i0 < end; i0 += kRemapAhead) {
    // entries past the row's end repeat its last one and are not added
    int c[kRemapAhead];
    double w[kRemapAhead], x[kRemapAhead][ND];
#pragma unroll
    for (int u = 0; u < kRemapAhead; ++u) {
      const int i = i0 + u < end ? i0 + u : end - 1;
      c[u] = col[i];
      w[u] = val[i];
    }
#pragma unroll
    for (int u = 0; u < kRemapAhead; ++u)
#pragma unroll
      for (int d = 0; d < ND; ++d) x[u][d] = s[(size_t)(d < nd ? d : 0) * nsend + c[u]];
#pragma unroll
    for (int u = 0; u < kRemapAhead; ++u) {
      if (i0 + u >= end) break;
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const double prod = x[u][d] * w[u];
        acc[d] = acc[d] + prod;
      }
    }
  }
#pragma unroll
  for (int d = 0; d < ND; ++d)
    if (d < nd) recv[(size_t)(d0 + d) * nrecv + r] = acc[d];
}

void remap_release(sht_remap *m) {
  if (m->row) (void)hipFree(m->row);
  if (m->col) (void)hipFree(m->col);
  if (m->val) (void)hipFree(m->val);
  delete m;
}

}  // namespace
}  // namespace sht

using namespace sht;

extern "C" {

int sht_remap_create(const int *send_index, const int *recv_index, const double *coef, int nnz,
                     int nsend, int nrecv, sht_remap **out) {
  if (!out) return fail(SHT_ERR_INVALID, "sht_remap_create: out is NULL");
  *out = nullptr;
  if (nnz < 0 || nsend < 1 || nrecv < 1 || (nnz > 0 && (!send_index || !recv_index || !coef)))
    return fail(SHT_ERR_INVALID, "sht_remap_create: bad sizes or NULL triplets");
  for (int i = 0; i < nnz; ++i)
    if (send_index[i] < 0 || send_index[i] >= nsend || recv_index[i] < 0 || recv_index[i] >= nrecv)
      return fail(SHT_ERR_INVALID, "sht_remap_create: index out of range at triplet " + std::to_string(i));
  // stable regrouping by receiving point keeps the reference's summation order
  std::vector<int> order(nnz);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return recv_index[a] < recv_index[b]; });
  std::vector<int> row(nrecv + 1, 0), col(nnz);
  std::vector<double> val(nnz);
  for (int i = 0; i < nnz; ++i) row[recv_index[i] + 1] += 1;
  for (int r = 0; r < nrecv; ++r) row[r + 1] += row[r];
  for (int i = 0; i < nnz; ++i) {
    col[i] = send_index[order[i]];
    val[i] = coef[order[i]];
  }
  sht_remap *m = new (std::nothrow) sht_remap;
  if (!m) return fail(SHT_ERR_NOMEM, "sht_remap_create: host allocation failed");
  m->nsend = nsend;
  m->nrecv = nrecv;
  m->nnz = nnz;
  const size_t nz = nnz > 0 ? (size_t)nnz : 1;
  if (hipMalloc(&m->row, sizeof(int) * (nrecv + 1)) != hipSuccess ||
      hipMalloc(&m->col, sizeof(int) * nz) != hipSuccess ||
      hipMalloc(&m->val, sizeof(double) * nz) != hipSuccess) {
    remap_release(m);
    return fail(SHT_ERR_NOMEM, "sht_remap_create: device allocation failed");
  }
  if (hipMemcpy(m->row, row.data(), sizeof(int) * (nrecv + 1), hipMemcpyHostToDevice) != hipSuccess ||
      (nnz > 0 && (hipMemcpy(m->col, col.data(), sizeof(int) * nnz, hipMemcpyHostToDevice) != hipSuccess ||
                   hipMemcpy(m->val, val.data(), sizeof(double) * nnz, hipMemcpyHostToDevice) != hipSuccess))) {
    remap_release(m);
    return fail(SHT_ERR_DEVICE, "sht_remap_create: upload failed");
  }
  *out = m;
  return SHT_OK;
}

void sht_remap_destroy(sht_remap *m) {
  if (m) remap_release(m);
}

int sht_remap_apply_dev(const sht_remap *m, const double *send, double *recv, int ndata, void *stream) {
  if (!m) return fail(SHT_ERR_INVALID, "sht_remap_apply_dev: remap is NULL");
  if (!send || !recv || ndata < 1) return fail(SHT_ERR_INVALID, "sht_remap_apply_dev: bad arguments");
  const int64_t n = (int64_t)m->nrecv * ndata;
  if (n > (int64_t)INT32_MAX * 128) return fail(SHT_ERR_INVALID, "sht_remap_apply_dev: too many outputs");
  // groups of 4 fields where that still gives each CU a workgroup
  const bool wide = (int64_t)m->nrecv * (ndata / 4) >= 256 * 256;
  const int64_t nt = wide ? (int64_t)m->nrecv * ((ndata + 3) / 4) : n;
  (wide ? remap_kernel<4> : remap_kernel<1>)<<<(unsigned)((nt + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      m->row, m->col, m->val, send, recv, m->nsend, m->nrecv, ndata);
  SHT_HIP(hipGetLastError());
  return SHT_OK;
}

}  // extern "C"
