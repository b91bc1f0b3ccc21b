// Operator renormalisation: CRS_CRS_CCS_PRODUCT (sml/CRS_CRS_CCS_PRODUCT.c:6-124), the
// product T^dagger O T that DMRG_TRANS_MAT_ONE/TWO/C_C apply to every block operator
// (dmrg/DMRG_TRANS_MAT_ONE.c:6-54 through DMRG_EXTEND_AND_REDUCE).
//
// The reference forms Out = M1 (M2 M3) in two passes, each entry a sum in a fixed order
// with entries of magnitude <= 1e-15 dropped:
//   pass 1  W(i, j)  = sum over the entries k of row i of M2, in stored order,
//                      of M3(col_k, j) * M2_k
//   pass 2  Out(i, j) = sum over the kept rows r of column j of W, ascending,
//                      of M1(i, r) * W(r, j)
// Here M3 is expanded to a dense device matrix, pass 1 is a CRS x dense product (one thread
// per entry of W, the row's entries in stored order, dropped entries set to 0), and pass 2
// is a CRS x dense product over the rows of M1 with their entries in ascending column
// order, skipping the zeros of W: the same nonzero terms in the same order as the
// reference's (the terms the reference adds for M1(i, r) = 0 are signed zeros, which do not
// change a sum).  The file is built without FMA contraction, so Out is the reference's bit
// for bit.  The dense result is compacted on the device.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "entry.h"

namespace dmrgx {
namespace {

constexpr double kDropBelow = 1e-15;

// dense[r][j] = M3(r, j) from CCS (col_ptr over columns, row indices per entry), one wavefront
// per column (Hubbard m = 396: 89 us with a thread per column, 7 with this).  serial: by its
// first lane alone, in stored order, for columns that hold a row twice (the last value stays).
__global__ __launch_bounds__(64) void k_ccs_to_dense(int32_t cols, const int64_t *__restrict__ cptr,
                                                     const int32_t *__restrict__ ridx, const double *__restrict__ val,
                                                     double *__restrict__ dense, int serial) {
  const int32_t j = blockIdx.x;
  const int step = serial ? 1 : 64;
  if (serial && threadIdx.x > 0) return;
  for (int64_t e = cptr[j] + threadIdx.x; e < cptr[j + 1]; e += step) dense[(int64_t)ridx[e] * cols + j] = val[e];
}

// out[i][j] = sum over the entries e of row i of A (stored order) of B[col_e][j] * A_e,
// dropped to 0 when |sum| <= 1e-15; with skip_zero, terms whose B value is 0 are left out.
// With kept set, the number of kept entries other than the last one, (rows-1, cols-1), is
// added to *kept (the count the reference's capacity check sees, CRS_CRS_CCS_PRODUCT.c:56);
// with row_kept set, every row's number of kept entries to row_kept[row].
// Waits for the loads of B, whose rows the entries pick: eight are in flight per thread, the
// sum stays in stored order (Hubbard m = 396, T^dagger O T: 46 -> 40 and 63 -> 29 us a pass).
template <bool kSkipZero>
__global__ __launch_bounds__(256) void k_crs_dense(int32_t rows, int32_t cols, const int64_t *__restrict__ rptr,
                                                   const int32_t *__restrict__ cidx, const double *__restrict__ aval,
                                                   const double *__restrict__ B, double *__restrict__ out,
                                                   unsigned long long *kept, int32_t *row_kept) {
  const int32_t j = blockIdx.x * 256 + threadIdx.x;
  const bool in = j < cols;
  const int32_t jj = in ? j : cols - 1;
  unsigned int mine = 0;
  for (int32_t i = blockIdx.y; i < rows; i += gridDim.y) {
    double s = 0.0;
    const int64_t e1 = rptr[i + 1];
    for (int64_t e = rptr[i]; e < e1; e += 8) {
      double b[8], a[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int64_t q = e + u < e1 ? e + u : e1 - 1;
        b[u] = B[(int64_t)cidx[q] * cols + jj];
        a[u] = aval[q];
      }
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (e + u < e1 && (!kSkipZero || b[u] != 0.0)) s = s + b[u] * a[u];
    }
    const bool keep = in && std::fabs(s) > kDropBelow;
    if (in) out[(int64_t)i * cols + j] = keep ? s : 0.0;
    if (keep && !(i == rows - 1 && j == cols - 1)) mine++;
    if (row_kept) {
      const int n = __popcll(__ballot(keep));
      if ((threadIdx.x & 63) == 0 && n) atomicAdd(row_kept + i, n);
    }
  }
  if (!kept) return;   // uniform over the launch
  __shared__ unsigned int cnt;
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  if (mine) atomicAdd(&cnt, mine);
  __syncthreads();
  if (threadIdx.x == 0 && cnt) atomicAdd(kept, (unsigned long long)cnt);
}

// Row pointers of the kept entries from their counts (one workgroup), and whether the last
// entry, (rows-1, cols-1), is kept: rptr[rows + 1].
__global__ __launch_bounds__(256) void k_row_pointers(int32_t rows, const int32_t *__restrict__ count,
                                                      const double *__restrict__ out, int64_t last, int64_t *rptr) {
  __shared__ int64_t sum[256];
  const int32_t per = (rows + 255) / 256, b = min((int32_t)threadIdx.x * per, rows), e = min(b + per, rows);
  int64_t mine = 0;
  for (int32_t i = b; i < e; i++) mine += count[i];
  sum[threadIdx.x] = mine;
  __syncthreads();
  int64_t at = 0;
  for (int t = 0; t < (int)threadIdx.x; t++) at += sum[t];
  for (int32_t i = b; i < e; i++) {
    rptr[i] = at;
    at += count[i];
  }
  if (threadIdx.x == 255) {
    rptr[rows] = at;
    rptr[rows + 1] = out[last] != 0.0;
  }
}

// The kept entries of the dense result, columns ascending: one wavefront per row.
__global__ __launch_bounds__(64) void k_compact_rows(int32_t rows, int32_t cols, const double *__restrict__ dense,
                                                     const int64_t *__restrict__ rptr, int32_t *__restrict__ col,
                                                     double *__restrict__ val) {
  for (int32_t i = blockIdx.x; i < rows; i += gridDim.x) {
    int64_t at = rptr[i];
    for (int32_t j0 = 0; j0 < cols; j0 += 64) {
      const int32_t j = j0 + threadIdx.x;
      const double v = j < cols ? dense[(int64_t)i * cols + j] : 0.0;
      const unsigned long long m = __ballot(v != 0.0);
      if (v != 0.0) {
        const int64_t q = at + __popcll(m & ((1ull << threadIdx.x) - 1));
        col[q] = j;
        val[q] = v;
      }
      at += __popcll(m);
    }
  }
}

void check_crs(const CRS1 *M, const char *what) {
  if (!M || !M->Row || M->row_dim < 0 || M->col_dim < 0) throw Failure(DMRGX_ERR_ARG, what);
  const int64_t nnz = M->Row[M->row_dim];
  if (nnz > 0 && (!M->Col || !M->Val)) throw Failure(DMRGX_ERR_ARG, what);
  for (int32_t r = 0; r < M->row_dim; r++)
    if (M->Row[r] < 0 || M->Row[r] > M->Row[r + 1]) throw Failure(DMRGX_ERR_ARG, what);
  for (int64_t e = 0; e < nnz; e++)
    if (M->Col[e] < 0 || M->Col[e] >= M->col_dim) throw Failure(DMRGX_ERR_ARG, what);
}

}  // namespace
}  // namespace dmrgx

using namespace dmrgx;

extern "C" {

void CRS_CRS_CCS_PRODUCT(CRS1 *M1, CRS1 *M2, CCS1 *M3, CRS1 *Out, CCS1 *Work, double *Work_Vec) {
  (void)Work_Vec;
  run_or_die("CRS_CRS_CCS_PRODUCT", [&] {
    if (!M1 || !M2 || !M3 || !Out || !Work) throw Failure(DMRGX_ERR_ARG, "NULL argument");
    // the reference's checks (sml/CRS_CRS_CCS_PRODUCT.c:8-28)
    if (M1->col_dim != M2->row_dim || M2->col_dim != M3->row_dim)
      throw Failure(DMRGX_ERR_ARG, "matrix dimensions do not chain");
    if (Work->max_col <= M3->col_dim) throw Failure(DMRGX_ERR_ARG, "Work has too few columns");
    if (Out->max_row <= M1->row_dim) throw Failure(DMRGX_ERR_ARG, "Out has too few rows");
    check_crs(M1, "M1 is not a valid CRS1");
    check_crs(M2, "M2 is not a valid CRS1");
    const int32_t n1 = M1->row_dim, n2 = M2->row_dim, n3 = M3->row_dim, k = M3->col_dim;
    if (!M3->Col || k < 0 || n3 < 0) throw Failure(DMRGX_ERR_ARG, "M3 is not a valid CCS1");
    const int64_t nnz3 = M3->Col[k];
    for (int32_t c = 0; c < k; c++)
      if (M3->Col[c] < 0 || M3->Col[c] > M3->Col[c + 1]) throw Failure(DMRGX_ERR_ARG, "M3 is not a valid CCS1");
    bool twice = false;   // a column of M3 that may hold a row twice
    for (int32_t c = 0; c < k; c++)
      for (int64_t e = M3->Col[c]; e < M3->Col[c + 1]; e++) {
        if (M3->Row[e] < 0 || M3->Row[e] >= n3) throw Failure(DMRGX_ERR_ARG, "M3 is not a valid CCS1");
        twice |= e > M3->Col[c] && M3->Row[e] <= M3->Row[e - 1];
      }
    Context &C = ctx();
    hipStream_t st = C.stream;
    // M1's rows in ascending column order (the order pass 2 adds them in); a column stored
    // twice in a row keeps its last value, as the reference's dense scatter of the row does
    const int64_t nnz2 = M2->Row[n2];
    bool sorted = true;
    for (int32_t r = 0; r < n1 && sorted; r++)
      for (int64_t e = M1->Row[r] + 1; e < M1->Row[r + 1]; e++)
        if (M1->Col[e] <= M1->Col[e - 1]) {
          sorted = false;
          break;
        }
    std::vector<int64_t> hr1, perm;
    std::vector<int32_t> c1;
    std::vector<double> v1;
    const int64_t *p1 = reinterpret_cast<const int64_t *>(M1->Row);
    const int32_t *q1 = M1->Col;
    const double *a1 = M1->Val;
    if (!sorted) {
      hr1.assign(n1 + 1, 0);
      for (int32_t r = 0; r < n1; r++) {
        const int64_t b = M1->Row[r], e = M1->Row[r + 1];
        perm.resize(e - b);
        std::iota(perm.begin(), perm.end(), b);
        std::stable_sort(perm.begin(), perm.end(), [&](int64_t x, int64_t y) { return M1->Col[x] < M1->Col[y]; });
        for (int64_t t = 0; t < e - b; t++) {
          if (t + 1 < e - b && M1->Col[perm[t + 1]] == M1->Col[perm[t]]) continue;
          c1.push_back(M1->Col[perm[t]]);
          v1.push_back(M1->Val[perm[t]]);
        }
        hr1[r + 1] = (int64_t)c1.size();
      }
      p1 = hr1.data();
      q1 = c1.data();
      a1 = v1.data();
    }
    const int64_t nd3 = (int64_t)n3 * k, nw = (int64_t)n2 * k, no = (int64_t)n1 * k;
    // the result's row pointers, whether its last entry is kept, the entries kept of W; then, on the
    // device behind them, its values and columns
    std::vector<int64_t> meta((size_t)n1 + 3, 0);
    const size_t meta_bytes = sizeof(int64_t) * meta.size();
    std::vector<char> all;   // a small result, copied back whole with its pointers
    DevBuf<char> mem, result;
    if (k > 0 && n1 > 0) {
      DevView<int64_t> r1, r2, p3;
      DevView<int32_t> dc1, dc2, dr3, count;
      DevView<double> dv1, dv2, dv3;
      const std::vector<int32_t> zeros(n1, 0);
      Upload up;
      up.add(r1, p1, (size_t)n1 + 1);
      up.add(dc1, q1, (size_t)p1[n1]);
      up.add(dv1, a1, (size_t)p1[n1]);
      up.add(r2, reinterpret_cast<const int64_t *>(M2->Row), (size_t)n2 + 1);
      up.add(dc2, M2->Col, (size_t)nnz2);
      up.add(dv2, M2->Val, (size_t)nnz2);
      up.add(p3, reinterpret_cast<const int64_t *>(M3->Col), (size_t)k + 1);
      up.add(dr3, M3->Row, (size_t)nnz3);
      up.add(dv3, M3->Val, (size_t)nnz3);
      up.add(count, zeros);
      up.place(mem);
      up.send();
      DevBuf<double> d3(nd3 > 0 ? nd3 : 1), w(nw > 0 ? nw : 1), o(no);
      result.resize(meta_bytes + (sizeof(double) + sizeof(int32_t)) * (size_t)no);
      int64_t *dmeta = reinterpret_cast<int64_t *>(result.p);
      double *oval = reinterpret_cast<double *>(result.p + meta_bytes);
      int32_t *ocol = reinterpret_cast<int32_t *>(oval + no);
      unsigned long long *dkept = reinterpret_cast<unsigned long long *>(dmeta + n1 + 2);
      HIPCHK(hipMemsetAsync(dkept, 0, sizeof(unsigned long long), st));
      if (nd3 > 0) HIPCHK(hipMemsetAsync(d3.p, 0, sizeof(double) * nd3, st));
      const unsigned gx = (unsigned)((k + 255) / 256);
      k_ccs_to_dense<<<k, 64, 0, st>>>(k, p3.p, dr3.p, dv3.p, d3.p, twice ? 1 : 0);
      // grid y at most 65535; the kernels loop over the rows beyond it
      if (n2 > 0)
        k_crs_dense<false><<<dim3(gx, (unsigned)std::min(n2, 65535)), 256, 0, st>>>(n2, k, r2.p, dc2.p, dv2.p, d3.p,
                                                                                   w.p, dkept, nullptr);
      k_crs_dense<true><<<dim3(gx, (unsigned)std::min(n1, 65535)), 256, 0, st>>>(n1, k, r1.p, dc1.p, dv1.p, w.p, o.p,
                                                                                nullptr, count.p);
      k_row_pointers<<<1, 256, 0, st>>>(n1, count.p, o.p, no - 1, dmeta);
      k_compact_rows<<<(unsigned)std::min(n1, 65535), 64, 0, st>>>(n1, k, o.p, dmeta, ocol, oval);
      HIPCHK(hipGetLastError());
      // small results: all of the buffer in one copy, rather than a wait for the count before a second
      // (Hubbard, a call in us, one copy and the parts: 63 KiB 79 and 91, 130 KiB 91 and 99, 231 KiB 106
      // and 107, 332 KiB 119 and 116, 831 KiB 195 and 180)
      if (result.count <= 256 * 1024) {
        all.resize(result.count);
        C.copy_out(all.data(), result.p, all.size());
        std::memcpy(meta.data(), all.data(), meta_bytes);
      } else {
        C.copy_out(meta.data(), result.p, meta_bytes);
      }
    }
    const long long w_kept = meta[n1 + 2];
    // The reference checks the kept count against the capacity before every entry it
    // evaluates (CRS_CRS_CCS_PRODUCT.c:56 for Work, :101 for Out), so it exits when the
    // entries kept before the last evaluated position reach max_val, even if nothing more
    // is stored after them.
    if (n2 > 0 && k > 0 && w_kept >= (long long)Work->max_val)
      throw Failure(DMRGX_ERR_ARG, "Work has too few elements");
    if (n1 > 0 && k > 0 && meta[n1] - meta[n1 + 1] >= (int64_t)Out->max_val)
      throw Failure(DMRGX_ERR_ARG, "Out has too few elements");
    if (meta[n1] > (int64_t)Out->max_val) throw Failure(DMRGX_ERR_ARG, "Out has too few elements");
    // Out, columns ascending (sml/CRS_CRS_CCS_PRODUCT.c:98-121)
    for (int32_t i = 0; i <= n1; i++) Out->Row[i] = (long)meta[i];
    const size_t nz = (size_t)meta[n1], col_at = meta_bytes + sizeof(double) * (size_t)no;
    if (nz > 0 && !all.empty()) {
      std::memcpy(Out->Val, all.data() + meta_bytes, sizeof(double) * nz);
      std::memcpy(Out->Col, all.data() + col_at, sizeof(int32_t) * nz);
    } else if (nz > 0) {
      C.copy_out(Out->Val, result.p + meta_bytes, sizeof(double) * nz);
      C.copy_out(Out->Col, result.p + col_at, sizeof(int32_t) * nz);
    }
    Out->row_dim = n1;
    Out->col_dim = k;
  });
}

}  // extern "C"
