// Operator update on the GPU: the stored 1D factor blocks of a kronmult
// handle rebuilt from dense 1D operator matrices that are already on the
// device, with no host copy of the blocks (update_kronmult_coefficients,
// src/asgard_kronmult_matrix.cpp:710-811).
//
// Sparse-grid and global handles store one n x n block per (connect_1d
// connection, term, dimension) in the vA layout [connection][term][dim][n*n]
// (make_kronmult_sparse, src/asgard_kronmult_matrix.cpp:369-393); dense
// handles store per term [dim][column block][row block][n*n].  Every block is
// column-major: entry (s, c) of the block of 1D cells (row, col) is
// A(n*row + s, n*col + c).  One thread per stored value; the reads are
// gathers from the operator matrices, the writes coalesced.
#include "akm_internal.hpp"
#include "grid.hpp"
#include "matrix.hpp"

#include <algorithm>
#include <limits>
#include <vector>

namespace akm
{
constexpr int op_threads = 256;

static int op_blocks(int64_t work)
{
  const int64_t b = (work + op_threads - 1) / op_threads;
  return static_cast<int>(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

//! vA[((j*T + t)*d + k)*n*n + c*n + s] = A_{t,k}(n*row_j + s, n*col_j + c).
template<typename P>
__global__ void __launch_bounds__(op_threads)
    gather_grid_blocks(const P *const *ops, int64_t lda, const int *conn_row, const int *conn_col,
                       int64_t nconn, int T, int d, int n, P *vA)
{
  const int nn = n * n;
  const int64_t total = nconn * T * d * nn;
  for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x)
  {
    const int q = static_cast<int>(idx % nn);
    int64_t rest = idx / nn;
    const int k = static_cast<int>(rest % d);
    rest /= d;
    const int t = static_cast<int>(rest % T);
    const int64_t j = rest / T;
    const int c = q / n, s = q - c * n;
    vA[idx] = ops[t * d + k][int64_t(n) * conn_row[j] + s + lda * (int64_t(n) * conn_col[j] + c)];
  }
}

//! The LDS-table copy of the factors: [dim][connection][term][nnp], the
//! padding of every block zero.
template<typename P>
__global__ void __launch_bounds__(op_threads)
    relayout_blocks(const P *vA, int64_t nconn, int T, int d, int n, int nnp, P *vAk)
{
  const int nn = n * n;
  const int64_t total = int64_t(d) * nconn * T * nnp;
  for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x)
  {
    const int q = static_cast<int>(idx % nnp);
    int64_t rest = idx / nnp;
    const int t = static_cast<int>(rest % T);
    rest /= T;
    const int64_t j = rest % nconn;
    const int k = static_cast<int>(rest / nconn);
    vAk[idx] = (q < nn) ? vA[((j * T + t) * d + k) * nn + q] : P(0);
  }
}

//! Dense handles, term t: term[((k*nb + ocol)*nb + orow)*n*n + c*n + s] =
//! A_{t,k}(n*orow + s, n*ocol + c) (src/asgard_kronmult_matrix.cpp:741-754).
template<typename P>
__global__ void __launch_bounds__(op_threads)
    gather_dense_blocks(const P *const *ops, int64_t lda, int nb, int d, int n, int t, P *term)
{
  const int nn = n * n;
  const int64_t total = int64_t(d) * nb * nb * nn;
  for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
       idx += int64_t(gridDim.x) * blockDim.x)
  {
    const int q = static_cast<int>(idx % nn);
    int64_t rest = idx / nn;
    const int orow = static_cast<int>(rest % nb);
    rest /= nb;
    const int ocol = static_cast<int>(rest % nb);
    const int k = static_cast<int>(rest / nb);
    const int c = q / n, s = q - c * n;
    term[idx] = ops[t * d + k][int64_t(n) * orow + s + lda * (int64_t(n) * ocol + c)];
  }
}

int relayout_factors(akm_matrix_s &m)
{
  const int64_t count = int64_t(m.d) * m.nconn * m.T * m.nnp;
  AKM_TRY(m.vAk.allocate(count * int64_t(m.esize)));
  auto go = [&](auto zero) {
    using P = decltype(zero);
    relayout_blocks<P><<<op_blocks(count), op_threads, 0, m.stream>>>(
        reinterpret_cast<const P *>(m.vA.data()), m.nconn, m.T, m.d, m.n, m.nnp,
        reinterpret_cast<P *>(m.vAk.data()));
  };
  if (m.prec == AKM_F64)
    go(0.0);
  else
    go(0.0f);
  return check_launch("LDS tables");
}

template<typename P>
static int update_operators_typed(akm_matrix_s &m, const void *const *ops_dev, int64_t lda)
{
  const P *const *ops = reinterpret_cast<const P *const *>(ops_dev);
  const int d = m.d, n = m.n, T = m.T;
  if (m.mode == mode_dense)
  {
    const int64_t work = int64_t(d) * m.nb * m.nb * n * n;
    for (int t = 0; t < T; t++)
    {
      gather_dense_blocks<P><<<op_blocks(work), op_threads, 0, m.stream>>>(
          ops, lda, m.nb, d, n, t, reinterpret_cast<P *>(m.terms[t].data()));
      AKM_TRY(check_launch("operator update (dense blocks)"));
    }
    return AKM_SUCCESS;
  }
  const int64_t nconn = (m.op_conn.size() - T * d - 1) / 2;
  P *vA = reinterpret_cast<P *>(m.vA.data());
  gather_grid_blocks<P><<<op_blocks(m.num_vA), op_threads, 0, m.stream>>>(
      ops, lda, m.op_conn.data(), m.op_conn.data() + nconn, nconn, T, d, n, vA);
  AKM_TRY(check_launch("operator update (factor blocks)"));
  if (m.mode == mode_grid && m.vAk.data() != nullptr)
    AKM_TRY(relayout_factors(m));
  if (m.mode == mode_global)
  {
    AKM_TRY(global_device_jacobi(m));
    AKM_TRY(global_tables(m));
  }
  return AKM_SUCCESS;
}

//! connect_1d on the device as (row, column) per connection, in vA order, and
//! after it the flags of scan_factors.
static int need_connections(akm_matrix_s &m)
{
  if (m.op_conn.size() > 0)
    return AKM_SUCCESS;
  std::vector<int> p1 = m.conn_pntr_host, i1 = m.conn_indx_host, dg;
  if (i1.empty())
    AKM_TRY(build_connect_1d(m.max_level, true, p1, i1, dg));
  const int64_t nconn = static_cast<int64_t>(i1.size());
  if (nconn * m.T * m.d * m.n * m.n != m.num_vA)
    return set_error(AKM_ERR_INVALID, "operator update: stored blocks do not match connect_1d");
  std::vector<int> rc(2 * nconn + m.T * m.d + 1, 0);
  for (int r = 0; r + 1 < static_cast<int>(p1.size()); r++)
    for (int j = p1[r]; j < p1[r + 1]; j++)
    {
      rc[j] = r;
      rc[nconn + j] = i1[j];
    }
  m.op_scan = 0;
  return m.op_conn.upload(rc.data(), int64_t(rc.size()), m.stream);
}

//! flags[t*d + k] = scan for a factor that is not exactly the identity (0 off
//! the diagonal blocks, the unit matrix on them), flags[T*d] = scan when any
//! value is not finite; the others keep a lower number.  A row of workgroups
//! per factor.
template<typename P>
__global__ void __launch_bounds__(op_threads)
    scan_factors(const P *vA, const int *conn_row, const int *conn_col, int64_t nconn, int pairs,
                 int n, int scan, int *flags)
{
  const int nn = n * n;
  for (int td = blockIdx.y; td < pairs; td += gridDim.y)
  {
    int other = 0, infinite = 0;
    for (int64_t i = blockIdx.x * int64_t(op_threads) + threadIdx.x; i < nconn * nn;
         i += int64_t(gridDim.x) * op_threads)
    {
      const int64_t q = i / nn;
      const int w = static_cast<int>(i - q * nn);
      const P v = vA[(q * pairs + td) * nn + w];
      const P unit = (conn_row[q] == conn_col[q] && w % (n + 1) == 0) ? P(1) : P(0);
      other |= (v != unit);
      infinite |= !isfinite(v);
    }
    other = __syncthreads_or(other);
    infinite = __syncthreads_or(infinite);
    if (threadIdx.x == 0 && other != 0)
      atomicMax(flags + td, scan);
    if (threadIdx.x == 0 && infinite != 0)
      atomicMax(flags + pairs, scan);
  }
}

int stored_factors(akm_matrix_s &m, std::vector<int> &mask, bool &finite)
{
  AKM_TRY(need_connections(m));
  const int pairs = m.T * m.d;
  const int64_t nconn = (m.op_conn.size() - pairs - 1) / 2;
  int *flags = m.op_conn.data() + 2 * nconn;
  if (m.op_scan == std::numeric_limits<int>::max())
  {
    AKM_HIP(hipMemsetAsync(flags, 0, sizeof(int) * (pairs + 1), m.stream));
    m.op_scan = 0;
  }
  const int scan = ++m.op_scan;
  // four values a thread, so that the 2.7 MB of a d = 6 level-7 operator of
  // six terms are read by 360 workgroups
  const dim3 grid(op_blocks((nconn * m.n * m.n + 3) / 4), std::min(pairs, 65535));
  const int *row = m.op_conn.data(), *col = row + nconn;
  if (m.prec == AKM_F64)
    scan_factors<double><<<grid, op_threads, 0, m.stream>>>(
        reinterpret_cast<const double *>(m.vA.data()), row, col, nconn, pairs, m.n, scan, flags);
  else
    scan_factors<float><<<grid, op_threads, 0, m.stream>>>(
        reinterpret_cast<const float *>(m.vA.data()), row, col, nconn, pairs, m.n, scan, flags);
  AKM_TRY(check_launch("factor scan"));
  mask.resize(pairs + 1);
  AKM_HIP(hipMemcpyAsync(mask.data(), flags, sizeof(int) * (pairs + 1), hipMemcpyDeviceToHost,
                         m.stream));
  AKM_HIP(hipStreamSynchronize(m.stream));
  for (int &f : mask)
    f = (f == scan) ? 1 : 0;
  finite = mask.back() == 0;
  mask.pop_back();
  return AKM_SUCCESS;
}

} // namespace akm

using namespace akm;

akm_status akm_update_operators(akm_matrix mat, const void *const *ops, int64_t lda)
{
  if (mat == nullptr)
    return set_error(AKM_ERR_INVALID, "operator update: null handle");
  if (mat->T == 0)
    return AKM_SUCCESS;
  if (ops == nullptr)
    return set_error(AKM_ERR_INVALID, "operator update: null operator list");
  mat->vA_stamp++;
  const int nops = mat->T * mat->d;
  for (int i = 0; i < nops; i++)
    if (ops[i] == nullptr)
      return set_error(AKM_ERR_INVALID, "operator update: operator %d is null", i);
  int64_t need = 0;
  if (mat->mode == mode_dense)
    need = int64_t(mat->n) * mat->nb;
  else if (mat->mode == mode_grid || mat->mode == mode_global)
    need = int64_t(mat->n) << mat->max_level;
  else
    return set_error(AKM_ERR_UNSUPPORTED,
                     "operator update: needs a sparse-grid, global or dense handle (this one "
                     "was made from an explicit index list)");
  if (lda < need)
    return set_error(AKM_ERR_INVALID, "operator update: lda %lld below the operator size %lld",
                     static_cast<long long>(lda), static_cast<long long>(need));
  if (mat->mode != mode_dense)
    AKM_TRY(need_connections(*mat));
  std::vector<const void *> ptrs(ops, ops + nops);
  AKM_TRY(mat->op_ptrs.upload(ptrs.data(), nops, mat->stream));
  if (mat->prec == AKM_F64)
    AKM_TRY(update_operators_typed<double>(*mat, mat->op_ptrs.data(), lda));
  else
    AKM_TRY(update_operators_typed<float>(*mat, mat->op_ptrs.data(), lda));
  if (mat->mode == mode_grid)
    AKM_TRY(factored_refresh(*mat));
  AKM_HIP(hipStreamSynchronize(mat->stream));
  return AKM_SUCCESS;
}
