// Device-resident restarted GMRES for the implicit (backward-Euler) step
// (I - dt*A) x = b.
//
// akm_gmres_euler is the algorithm of solver::simple_gmres
// (src/solver.cpp:156-298) with every vector and Hessenberg operation on the
// GPU.  An inner iteration is the fused apply (kronmult + identity) and two
// kernels: the classical Gram-Schmidt dot products V^T w, and the update
// w -= V h with the partial sums of |w|^2.  What only needs those sums (the
// norm, the rotation of the Hessenberg column and of the right-hand side with
// reference BLAS rot/rotg semantics, the residual estimate) is done by an
// extra workgroup of the next step's dot products, beside them, and stored
// straight to pinned host memory.  A Krylov vector stays as the update leaves
// it, with its 1/norm kept aside: the operator is linear, so the factor goes
// into the next step's coefficients and no pass scales vectors (except for
// preconditioned directions, which may be nonlinear).  Reductions use fixed
// partitions and orders, so results repeat bit for bit.  The host reads one
// scalar per iteration to test convergence.
//
// What bounds a step at 64,768 unknowns: the latency of its three dependent
// launches, 8.5 (apply) + 4.8 + 6.2 us.  One kernel each for the dots, the
// reduction and update, the Givens step with the scaling, and a copy of the
// state to the host took 8.4 + 10.6 + 4.8 + 2.7 us beside the apply; letting
// the update's last workgroup finish the step took 14.2 us for the update
// (the tail of device-scope accesses is serial).
//
// akm_gmres_euler_mixed is an FP64 iterative refinement around flexible
// GMRES cycles: the residual b - (I - dt*A)x, the Krylov basis, the
// Gram-Schmidt and the Hessenberg least squares are FP64; the operator inside
// a cycle may be the FP32 kronmult (vectors rounded to FP32 for the apply
// only) and a right preconditioner may act on every basis vector.  After each
// cycle the true FP64 residual decides: it must at least halve, else the
// cycle is undone and plain FP64 GMRES finishes the solve.
#include "matrix.hpp"
#include "precond.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <limits>
#include <mutex>
#include <vector>

namespace akm
{
constexpr int gm_threads = 256;
constexpr int gm_cols = 4; // Krylov columns per dot-product block
// the update's parts: columns are split over gm_split threads per row
constexpr int gm_split = 4;
constexpr int gm_tile = 128; // rows of an update block at a time
constexpr int gm_upd_threads = gm_split * gm_tile;
constexpr int gm_lanes = 8; // lanes that add one column's dot partials
// finishing a step stages 3 * restart values in LDS (64 KB)
constexpr int gm_max_restart = 2000;
// host copies of the step state: Arnoldi steps in flight at once (the step
// waited for plus the speculative ones) stay below this
constexpr int gm_slots = 8;
// speculative steps enqueued past the one waited for: one step on the GPU
// (about 15 us at d=4) covers the host's poll and its three launches
constexpr int gm_ahead = 1;

template<typename P>
struct gm_state
{
  P nrm;       // norm of the last orthogonalised vector
  P inner_res; // residual estimate |s_j g_j|
  P pad[2];
};

//! What the host reads of a step, in pinned memory: the value and the value
//! xor the step's number, so that the two stores need no order between them.
struct gm_host_state
{
  uint64_t value, check;
  uint64_t pad[6];
};

//! A step's scalar to the host (nothing when there is no slot).
__device__ __forceinline__ void gm_publish(gm_host_state *hs, double value, uint64_t seq)
{
  if (hs == nullptr)
    return;
  const uint64_t bits = static_cast<uint64_t>(__double_as_longlong(value));
  __hip_atomic_store(&hs->value, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&hs->check, bits ^ seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template<typename P>
__device__ __forceinline__ P block_sum(P v, P *sh)
{
  // fixed-order block reduction (deterministic): a shuffle tree inside each
  // wavefront, then the wavefronts' sums in order; two barriers
#pragma unroll
  for (int off = wave_size / 2; off > 0; off >>= 1)
    v += __shfl_xor(v, off, wave_size);
  const int wave = threadIdx.x / wave_size;
  if (threadIdx.x % wave_size == 0)
    sh[wave] = v;
  __syncthreads();
  P r = 0;
  for (int w = 0; w < static_cast<int>(blockDim.x) / wave_size; w++)
    r += sh[w];
  __syncthreads();
  return r;
}

template<typename P>
__device__ __forceinline__ void dev_rot(P &x, P &y, P c, P s)
{
  const P t = c * x + s * y;
  y = c * y - s * x;
  x = t;
}

//! reference BLAS rotg: r = +-sqrt(a^2+b^2) with the sign of the larger
//! magnitude entry, c = a/r, s = b/r; a <- r.
template<typename P>
__device__ __forceinline__ void dev_rotg(P &a, P b, P &c, P &s)
{
  const P roe = (fabs(a) > fabs(b)) ? a : b;
  const P scale = fabs(a) + fabs(b);
  if (scale == P{0})
  {
    c = 1;
    s = 0;
    a = 0;
    return;
  }
  const P as = a / scale, bs = b / scale;
  P r = scale * sqrt(as * as + bs * bs);
  r = (roe >= P{0}) ? r : -r;
  c = a / r;
  s = b / r;
  a = r;
}

//! What finishing a step reads and writes: the step's |w|^2 partials and
//! Hessenberg column h, the rotations, the right-hand side, and the state.
template<typename P>
struct gm_arrays
{
  P *h, *H, *cs, *sn, *g; // column, packed columns, rotations, right-hand side
  P *inv;                 // 1/norm of every stored Krylov vector; null: all unit
  P *sqp;                 // |w|^2 partials
  gm_state<P> *st;
};

//! The step an extra workgroup finishes: column j (-1: the start of a cycle,
//! where the norm is that of the residual), or nothing (count 0).
template<typename P>
struct gm_pending
{
  int j, count; // count: |w|^2 partials
  P tol;
  int rotate_always;
  gm_host_state *hs;
  uint64_t seq;
};

//! Finishes a step in one workgroup (see the file comment).  With j < 0:
//! g_0 = |r|.  Otherwise the old rotations down column j, the new one, the
//! residual estimate and the rotation of g, which with rotate_always == 0
//! happens only while the estimate is above tol, as simple_gmres does
//! (src/solver.cpp:261-267).  `lds`: 3 (j + 1) values.
template<typename P>
__device__ __forceinline__ void gm_finish_step(gm_arrays<P> const &a, gm_pending<P> const &p,
                                               P *lds, P *sh)
{
  const int j = p.j, t = threadIdx.x;
  P *lc = lds, *lcs = lds + (j + 1), *lsn = lcs + (j + 1);
  for (int k = t; k <= j; k += blockDim.x)
    lc[k] = a.h[k];
  for (int k = t; k < j; k += blockDim.x)
  {
    lcs[k] = a.cs[k];
    lsn[k] = a.sn[k];
  }
  const P gj = (j >= 0) ? a.g[j] : P{0};
  P s = 0;
#pragma unroll 4
  for (int b = t; b < p.count; b += blockDim.x)
    s += a.sqp[b];
  s = block_sum(s, sh); // its barriers also order the LDS writes above
  const P nrm = sqrt(s);
  if (t == 0)
  {
    P res = nrm;
    if (j < 0)
      a.g[0] = nrm;
    else
    {
      // down the column, the running entry in a register
      P x = lc[0];
      for (int k = 0; k < j; k++)
      {
        P y = lc[k + 1];
        dev_rot(x, y, lcs[k], lsn[k]);
        lc[k] = x;
        x = y;
      }
      P c, sv;
      dev_rotg(x, nrm, c, sv);
      lc[j] = x;
      a.cs[j] = c;
      a.sn[j] = sv;
      res = fabs(sv * gj);
      if (p.rotate_always != 0 || res > p.tol)
      {
        P u = gj, v = 0;
        dev_rot(u, v, c, sv);
        a.g[j] = u;
        a.g[j + 1] = v;
      }
    }
    gm_publish(p.hs, static_cast<double>(res), p.seq);
    a.st->nrm = nrm;
    a.st->inner_res = res;
    if (a.inv != nullptr)
      a.inv[j + 1] = (nrm > P{0}) ? P{1} / nrm : P{0};
  }
  __syncthreads();
  for (int k = t; k <= j; k += blockDim.x)
    a.H[(j * (j + 1)) / 2 + k] = lc[k]; // packed upper triangle, column j
}

//! gm_finish_step alone (the host waits for it before the next step is
//! enqueued).  Dynamic LDS: 3 (j + 1) values.
template<typename P>
__global__ void __launch_bounds__(gm_threads) gm_finish(gm_arrays<P> a, gm_pending<P> p)
{
  __shared__ P sh[gm_threads / wave_size];
  extern __shared__ unsigned char gf_raw[];
  gm_finish_step(a, p, reinterpret_cast<P *>(gf_raw), sh);
}

//! sqp[bx] = sum of x^2 over the block's rows (x is only read).
template<typename P>
__global__ void __launch_bounds__(gm_threads)
gm_sumsq(int64_t n, int64_t rows_per_block, const P *x, P *sqp)
{
  __shared__ P sh[gm_threads / wave_size];
  const int64_t r0 = blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  P sq = 0;
#pragma unroll 4
  for (int64_t i = r0 + threadIdx.x; i < r1; i += gm_threads)
  {
    const P v = x[i];
    sq = fma(v, v, sq);
  }
  sq = block_sum(sq, sh);
  if (threadIdx.x == 0)
    sqp[blockIdx.x] = sq;
}

//! partial[k*ndot + bx] = sum over rows of block bx of V_k[i] * w[i],
//! for k in [k0, k0 + gm_cols) intersect [0, ncols).  The wavefront reduces
//! its gm_cols sums together: each exchange halves the columns a lane holds.
//! Workgroup (ndot, 0) finishes the step before instead (pend.count > 0;
//! dynamic LDS: 3 (pend.j + 1) values).
template<typename P>
__global__ void __launch_bounds__(gm_threads)
gm_dots(int64_t n, int64_t rows_per_block, const P *V, int64_t ldv, const P *w, int ncols,
        int ndot, P *partial, gm_arrays<P> arr, gm_pending<P> pend)
{
  static_assert(gm_cols == 4, "the exchange below halves four columns twice");
  __shared__ P sh[gm_threads / wave_size][gm_cols];
  extern __shared__ unsigned char gd_raw[];
  if (static_cast<int>(blockIdx.x) == ndot)
  {
    if (blockIdx.y == 0)
      gm_finish_step(arr, pend, reinterpret_cast<P *>(gd_raw), &sh[0][0]);
    return;
  }
  const int64_t r0 = blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  const int k0 = blockIdx.y * gm_cols;
  P acc[gm_cols];
  const P *col[gm_cols];
#pragma unroll
  for (int c = 0; c < gm_cols; c++)
  {
    acc[c] = 0;
    // columns past the last repeat it; their sums are dropped
    col[c] = V + int64_t(min(k0 + c, ncols - 1)) * ldv;
  }
#pragma unroll 4
  for (int64_t i = r0 + threadIdx.x; i < r1; i += gm_threads)
  {
    const P wi = w[i];
#pragma unroll
    for (int c = 0; c < gm_cols; c++)
      acc[c] = fma(col[c][i], wi, acc[c]);
  }
  const int lane = threadIdx.x % wave_size;
  const bool up = (lane & 32) != 0, odd = (lane & 16) != 0;
  // lanes below 32 keep columns 0 and 1, the others 2 and 3; then one each
  const P a0 = (up ? acc[2] : acc[0]) + __shfl_xor(up ? acc[0] : acc[2], 32, wave_size);
  const P a1 = (up ? acc[3] : acc[1]) + __shfl_xor(up ? acc[1] : acc[3], 32, wave_size);
  P v = (odd ? a1 : a0) + __shfl_xor(odd ? a0 : a1, 16, wave_size);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1)
    v += __shfl_xor(v, off, wave_size);
  if ((lane & 15) == 0)
    sh[threadIdx.x / wave_size][(up ? 2 : 0) + (odd ? 1 : 0)] = v;
  __syncthreads();
  if (threadIdx.x < gm_cols && k0 + static_cast<int>(threadIdx.x) < ncols)
  {
    P s = 0;
#pragma unroll
    for (int w2 = 0; w2 < gm_threads / wave_size; w2++)
      s += sh[w2][threadIdx.x];
    partial[int64_t(k0 + threadIdx.x) * ndot + blockIdx.x] = s;
  }
}

//! Arnoldi step j after the dots (ndot partials per column): h, then
//! w <- w / |v_j| - V h with the |w|^2 partials; columns split over gm_split
//! threads per row.  Block 0 stores h.  Dynamic LDS: j + 1 values.
template<typename P>
__global__ void __launch_bounds__(gm_upd_threads)
gm_update(int64_t n, int64_t rows_per_block, const P *V, int64_t ldv, P *w, int j,
          const P *dotp, int ndot, gm_arrays<P> a)
{
  __shared__ P red[gm_split][gm_tile];
  __shared__ P sh[gm_upd_threads / wave_size];
  extern __shared__ unsigned char up_raw[];
  P *cf = reinterpret_cast<P *>(up_raw); // h_k / |stored v_k|
  const int t = threadIdx.x, ncols = j + 1;
  const P invj = (a.inv != nullptr) ? a.inv[j] : P{1};
  // gm_lanes lanes add one column's partials, the same order in every block
  for (int k = t / gm_lanes; k < ncols; k += gm_upd_threads / gm_lanes)
  {
    const P ik = (a.inv != nullptr) ? a.inv[k] : P{1};
    P v = 0;
#pragma unroll 8
    for (int b = t % gm_lanes; b < ndot; b += gm_lanes)
      v += dotp[int64_t(k) * ndot + b];
#pragma unroll
    for (int off = gm_lanes / 2; off > 0; off >>= 1)
      v += __shfl_xor(v, off, wave_size);
    if (t % gm_lanes == 0)
    {
      const P h = v * ik * invj;
      cf[k] = h * ik;
      if (blockIdx.x == 0)
        a.h[k] = h;
    }
  }
  __syncthreads();
  const int part = t / gm_tile, lane = t % gm_tile;
  const int64_t r0 = blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  P sq = 0;
  for (int64_t base = r0; base < r1; base += gm_tile)
  {
    const int64_t i = base + lane;
    P s = 0;
    if (i < r1)
    {
#pragma unroll 8
      for (int k = part; k < ncols; k += gm_split)
        s = fma(V[int64_t(k) * ldv + i], cf[k], s);
    }
    red[part][lane] = s;
    __syncthreads();
    if (part == 0 && i < r1)
    {
      P sum = red[0][lane];
#pragma unroll
      for (int q = 1; q < gm_split; q++)
        sum += red[q][lane];
      const P v = fma(w[i], invj, -sum);
      w[i] = v;
      sq = fma(v, v, sq);
    }
    __syncthreads();
  }
  sq = block_sum(sq, sh);
  if (t == 0)
    a.sqp[blockIdx.x] = sq;
}

//! w /= |w| (the norm of the state), for vectors a nonlinear map reads.
template<typename P>
__global__ void __launch_bounds__(gm_threads) gm_scale(int64_t n, P *w, const gm_state<P> *st)
{
  const P nrm = st->nrm;
  if (!(nrm > P{0}))
    return;
  const P inv = P{1} / nrm;
  for (int64_t i = blockIdx.x * int64_t(gm_threads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * gm_threads)
    w[i] *= inv;
}

//! Packed upper-triangular back-solve H y = g (tpsv 'U','N','N') in g, then
//! y_k / |stored v_k|.  One wavefront with an entry per lane for m <= 64
//! (no barriers: 11 us became 4 at m = 35); else one workgroup, g (and H when
//! it fits, `h_in_lds`) in LDS, the updates of one column over the threads.
//! The same operations in the same order per entry as a serial solve.
template<typename P>
__global__ void __launch_bounds__(64) gm_backsolve_wave(int m, const P *H, P *g, const P *inv)
{
  __shared__ P lh[64 * 65 / 2];
  const int lane = threadIdx.x;
#pragma unroll 8
  for (int i = lane; i < m * (m + 1) / 2; i += 64)
    lh[i] = H[i];
  P v = (lane < m) ? g[lane] : P{0};
  __syncthreads();
  const P own = (lane < m) ? lh[lane + (lane * (lane + 1)) / 2] : P{0};
  for (int j = m - 1; j >= 0; j--)
  {
    const P hij = (lane < j) ? lh[lane + (j * (j + 1)) / 2] : P{0};
    // every lane divides by its own diagonal, lane j's quotient counts.  A
    // zero diagonal only follows an exact breakdown (residual already zero);
    // that column then takes no part in the solution
    const P q = (own != P{0}) ? v / own : P{0};
    const P gj = __shfl(q, j, wave_size);
    if (lane < j)
      v -= gj * hij;
    else if (lane == j)
      v = gj;
  }
  if (lane < m)
    g[lane] = (inv != nullptr) ? v * inv[lane] : v;
}

template<typename P>
__global__ void __launch_bounds__(256)
gm_backsolve(int m, const P *H, P *g, int h_in_lds, const P *inv)
{
  extern __shared__ unsigned char bs_raw[];
  P *lg = reinterpret_cast<P *>(bs_raw);
  P *lh = lg + m;
  const int tid = threadIdx.x;
  for (int i = tid; i < m; i += 256)
    lg[i] = g[i];
  if (h_in_lds)
    for (int i = tid; i < m * (m + 1) / 2; i += 256)
      lh[i] = H[i];
  __syncthreads();
  const P *Hs = h_in_lds ? lh : H;
  for (int j = m - 1; j >= 0; j--)
  {
    if (tid == 0)
    {
      const P hjj = Hs[j + (j * (j + 1)) / 2];
      lg[j] = (hjj != P{0}) ? lg[j] / hjj : P{0};
    }
    __syncthreads();
    const P gj = lg[j];
    for (int i = tid; i < j; i += 256)
      lg[i] -= gj * Hs[i + (j * (j + 1)) / 2];
    __syncthreads();
  }
  for (int i = tid; i < m; i += 256)
    g[i] = (inv != nullptr) ? lg[i] * inv[i] : lg[i];
}

//! x += V[:, 0:m] y, the columns split over gm_split threads per row.
template<typename P>
__global__ void __launch_bounds__(gm_upd_threads)
gm_xupdate(int64_t n, int64_t rows_per_block, const P *V, int64_t ldv, int m, const P *y, P *x)
{
  __shared__ P red[gm_split][gm_tile];
  extern __shared__ unsigned char ys_raw[];
  P *ys = reinterpret_cast<P *>(ys_raw);
  for (int k = threadIdx.x; k < m; k += gm_upd_threads)
    ys[k] = y[k];
  __syncthreads();
  const int part = threadIdx.x / gm_tile, lane = threadIdx.x % gm_tile;
  const int64_t r0 = blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  for (int64_t base = r0; base < r1; base += gm_tile)
  {
    const int64_t i = base + lane;
    P s = 0;
    if (i < r1)
    {
#pragma unroll 8
      for (int k = part; k < m; k += gm_split)
        s = fma(V[int64_t(k) * ldv + i], ys[k], s);
    }
    red[part][lane] = s;
    __syncthreads();
    if (part == 0 && i < r1)
    {
      P sum = red[0][lane];
#pragma unroll
      for (int q = 1; q < gm_split; q++)
        sum += red[q][lane];
      x[i] += sum;
    }
    __syncthreads();
  }
}

//! r = b - r
template<typename P>
__global__ void __launch_bounds__(gm_threads) gm_rsub(int64_t n, const P *b, P *r)
{
  for (int64_t i = blockIdx.x * int64_t(gm_threads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * gm_threads)
    r[i] = b[i] - r[i];
}

//! y = fp32(scale * x)
__global__ void __launch_bounds__(gm_threads)
gm_to_f32(int64_t n, const double *x, double scale, float *y)
{
  for (int64_t i = blockIdx.x * int64_t(gm_threads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * gm_threads)
    y[i] = static_cast<float>(scale * x[i]);
}

//! Residual norms between which a residual goes into FP32 as it is: entries
//! and products a factor of 1e26 away from its norm still have all their bits.
constexpr double gm_f32_least = 1e-12, gm_f32_most = 1e12;

//! The power of two that brings a norm near one; 1 when it needs none.
static double f32_scale(double norm)
{
  if ((norm >= gm_f32_least && norm <= gm_f32_most) || !std::isfinite(norm) || norm == 0.0)
    return 1.0;
  return std::ldexp(1.0, -std::clamp(std::ilogb(norm), -1000, 1000));
}

//! w = v + c * y, y in FP32 (the identity part of I - dt*A stays FP64).
__global__ void __launch_bounds__(gm_threads)
gm_axpy_f32(int64_t n, const double *v, double c, const float *y, double *w)
{
  for (int64_t i = blockIdx.x * int64_t(gm_threads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * gm_threads)
    w[i] = fma(c, static_cast<double>(y[i]), v[i]);
}

//! y = alpha*A*x + beta*y for a dense n x n column-major A, one thread per
//! row (consecutive threads read consecutive entries of a column); beta == 0
//! never reads y.
template<typename P>
__global__ void __launch_bounds__(gm_threads)
gm_dense_gemv(int n, const P *A, const P *x, P alpha, P beta, P *y)
{
  const int i = blockIdx.x * gm_threads + threadIdx.x;
  if (i >= n)
    return;
  P s = 0;
  for (int j = 0; j < n; j++)
    s = fma(A[int64_t(j) * n + i], x[j], s);
  y[i] = (beta == P{0}) ? alpha * s : fma(alpha, s, beta * y[i]);
}

//! v = M^-1 v from the LU factors of M with partial pivoting (getrs after
//! getrf): the row interchanges piv in order, then the unit lower and the
//! upper triangular solves, column by column.  One workgroup, v in LDS.
template<typename P>
__global__ void __launch_bounds__(256) gm_lu_solve(int n, const P *LU, const int *piv, P *v)
{
  extern __shared__ unsigned char lu_raw[];
  P *lv = reinterpret_cast<P *>(lu_raw);
  const int tid = threadIdx.x;
  for (int i = tid; i < n; i += 256)
    lv[i] = v[i];
  __syncthreads();
  if (tid == 0)
    for (int k = 0; k < n; k++)
    {
      const int p = piv[k];
      if (p != k)
      {
        const P t = lv[k];
        lv[k] = lv[p];
        lv[p] = t;
      }
    }
  __syncthreads();
  for (int k = 0; k < n; k++)
  {
    const P vk = lv[k];
    for (int i = k + 1 + tid; i < n; i += 256)
      lv[i] -= LU[int64_t(k) * n + i] * vk;
    __syncthreads();
  }
  for (int k = n - 1; k >= 0; k--)
  {
    if (tid == 0)
      lv[k] /= LU[int64_t(k) * n + k];
    __syncthreads();
    const P vk = lv[k];
    for (int i = tid; i < k; i += 256)
      lv[i] -= LU[int64_t(k) * n + i] * vk;
    __syncthreads();
  }
  for (int i = tid; i < n; i += 256)
    v[i] = lv[i];
}

} // namespace akm

//! Device workspace of the solvers, kept with the matrix between solves.
struct akm_gmres_workspace
{
  int restart = 0;
  int64_t n = 0;
  size_t esize = 8;
  akm::dev_buffer<unsigned char> V, work, xb;
  akm::dev_buffer<unsigned char> state;
  // flexible / mixed-precision solver only
  akm::dev_buffer<double> Z, xprev;
  akm::dev_buffer<float> v32, y32;
  akm::gm_host_state *host_state = nullptr; // pinned, gm_slots slots
  uint64_t seq = 0;                         // step numbers given out so far
  ~akm_gmres_workspace()
  {
    if (host_state != nullptr)
      (void)hipHostFree(host_state);
  }
};

static void delete_workspace(akm_gmres_workspace *w) { delete w; }

namespace akm
{
//! Rows of a dot-product (and norm) block: four per thread, more past 512
//! blocks, so the per-column partial sums stay short.
static int64_t dot_rows(int64_t n) { return std::max<int64_t>(1024, (n + 511) / 512); }
//! Rows of an update block: one tile, more past 1024 blocks.
static int64_t update_rows(int64_t n)
{
  return std::max<int64_t>(1, (n + 1024 * gm_tile - 1) / (1024 * gm_tile)) * gm_tile;
}

//! Arnoldi steps are enqueued one ahead of the host's convergence check when
//! the operator apply takes less than this (milliseconds).
constexpr double speculate_below_ms = 0.25;

//! Runs f (which enqueues work on s) and measures it with HIP events.
template<typename F>
static int timed_on_stream(hipStream_t s, F &&f, double &ms)
{
  hipEvent_t e0, e1;
  AKM_HIP(hipEventCreate(&e0));
  AKM_HIP(hipEventCreate(&e1));
  int rc = AKM_SUCCESS;
  if (hipEventRecord(e0, s) != hipSuccess)
    rc = set_error(AKM_ERR_HIP, "gmres: event record failed");
  if (rc == AKM_SUCCESS)
    rc = f();
  float t = 0;
  if (rc == AKM_SUCCESS &&
      (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
       hipEventElapsedTime(&t, e0, e1) != hipSuccess))
    rc = set_error(AKM_ERR_HIP, "gmres: event timing failed");
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  ms = t;
  return rc;
}

//! Memory of one solve: the Krylov basis V (n x (restart + 1)), the small
//! work array (h, packed H, cs, sn, g, 1/norms, dot and norm partials:
//! gm_work_values of them), the device step state, and gm_slots pinned host
//! slots with the number of steps published to them, or one plain host state
//! (the host then waits for the whole stream).  Every value on the device is
//! written by a kernel before any kernel or the host reads it, so none needs
//! clearing between solves.
struct gm_memory
{
  void *V = nullptr;
  void *work = nullptr;
  void *state = nullptr;
  gm_host_state *slots = nullptr;
  uint64_t *seq = nullptr;
  void *host_state = nullptr;
};

//! Values in the small work array of a solve.
static int64_t gm_work_values(int64_t n, int restart)
{
  // sized for 256-row partials of every column, more than those in use
  // (dot_rows, update_rows) and the 1/norms take
  const int64_t rpb = std::max<int64_t>(256, (n + 1023) / 1024);
  const int64_t nblk = (n + rpb - 1) / rpb;
  const int64_t columns = int64_t(restart) * (restart + 1) / 2;
  const int64_t ndot = (n + dot_rows(n) - 1) / dot_rows(n);
  const int64_t nupd = (n + update_rows(n) - 1) / update_rows(n);
  return std::max(4 * int64_t(restart + 2) + columns + 2 + int64_t(restart + 1) * nblk + nblk + 16,
                  5 * int64_t(restart + 2) + columns + 2 + int64_t(restart + 1) * ndot +
                      std::max(nupd, ndot));
}

//! The memory of a solve in a matrix's workspace.
static gm_memory memory_of(akm_gmres_workspace &ws)
{
  gm_memory mem;
  mem.V = ws.V.data();
  mem.work = ws.work.data();
  mem.state = ws.state.data();
  mem.slots = ws.host_state;
  mem.seq = &ws.seq;
  return mem;
}

//! One restart cycle's device state and the kernel sequence of its steps.
template<typename P>
struct gm_cycle
{
  int64_t n = 0;
  hipStream_t s = nullptr;
  int restart = 0;
  P *V = nullptr;
  P *Z = nullptr; // preconditioned directions (flexible GMRES), else null
  int64_t ldv = 0;
  int64_t drows = 0, urows = 0;
  int ndot = 0, nupd = 0, sblocks = 0;
  P *h = nullptr, *H = nullptr, *cs = nullptr, *sn = nullptr, *g = nullptr, *inv = nullptr;
  P *dotp = nullptr, *sqp = nullptr;
  gm_state<P> *st = nullptr, *hst = nullptr;
  gm_host_state *slots = nullptr;
  uint64_t *seq = nullptr;
  uint64_t start_seq = 0; // number of the cycle's start, step j is start + 1 + j
  int finished = -2;      // last step finished by a launch (-1: the start)
  bool lazy = true; // Krylov vectors stored beside their 1/norm
  int rotate_always = 0;

  gm_cycle(gm_memory const &mem, int64_t n_, hipStream_t s_, int restart_, P *Z_,
           int rotate_always_)
      : n(n_), s(s_), restart(restart_), Z(Z_), rotate_always(rotate_always_)
  {
    V = static_cast<P *>(mem.V);
    ldv = n;
    drows = dot_rows(n);
    ndot = static_cast<int>((n + drows - 1) / drows);
    urows = update_rows(n);
    nupd = static_cast<int>((n + urows - 1) / urows);
    sblocks = static_cast<int>(std::min<int64_t>((n + gm_threads - 1) / gm_threads, 2048));
    // small work arrays: h, H (packed), cs, sn, g, 1/norms, dot and norm partials
    h = static_cast<P *>(mem.work);
    H = h + (restart + 1);
    cs = H + int64_t(restart) * (restart + 1) / 2 + 1;
    sn = cs + (restart + 1);
    g = sn + (restart + 1);
    inv = g + (restart + 2);
    dotp = inv + (restart + 2);
    sqp = dotp + int64_t(restart + 1) * ndot;
    st = static_cast<gm_state<P> *>(mem.state);
    hst = static_cast<gm_state<P> *>(mem.host_state);
    slots = mem.slots;
    seq = mem.seq;
  }

  gm_arrays<P> arrays() const
  {
    return gm_arrays<P>{h, H, cs, sn, g, lazy ? inv : nullptr, sqp, st};
  }

  //! Step j (-1: the start) as the kernel that finishes it sees it.
  gm_pending<P> pending(int j, P tol) const
  {
    const uint64_t number = start_seq + 1 + j;
    return gm_pending<P>{j,   (j < 0) ? ndot : nupd, tol, rotate_always,
                         (slots != nullptr) ? slots + number % gm_slots : nullptr, number};
  }

  //! Finishes step j in a launch of its own.
  int finish_step(int j, P tol)
  {
    gm_finish<P><<<1, gm_threads, 3 * sizeof(P) * (j + 1), s>>>(arrays(), pending(j, tol));
    finished = j;
    return check_launch("gmres step");
  }

  //! Waits until step j (-1: the start) is finished; res = its estimate.
  //! Polls the pinned slot the kernel writes; a stream that has run dry
  //! without writing it has failed.
  int wait_step(int j, P &res)
  {
    if (slots == nullptr)
    {
      AKM_HIP(hipMemcpyAsync(hst, st, sizeof(gm_state<P>), hipMemcpyDeviceToHost, s));
      AKM_HIP(hipStreamSynchronize(s));
      res = hst->inner_res;
      return AKM_SUCCESS;
    }
    const uint64_t number = start_seq + 1 + j;
    const gm_host_state *slot = slots + number % gm_slots;
    uint64_t value = 0;
    auto arrived = [&]() {
      value = __atomic_load_n(&slot->value, __ATOMIC_ACQUIRE);
      return (value ^ __atomic_load_n(&slot->check, __ATOMIC_ACQUIRE)) == number;
    };
    for (unsigned spin = 1; !arrived(); spin++)
    {
      if (spin % 4096 != 0)
      {
        __builtin_ia32_pause();
        continue;
      }
      const hipError_t e = hipStreamQuery(s);
      (void)hipGetLastError();
      if (e != hipErrorNotReady && (e != hipSuccess || !arrived()))
        return set_error(AKM_ERR_HIP, "gmres: step state not written: %s",
                         hipGetErrorString(e));
    }
    double v;
    std::memcpy(&v, &value, sizeof(v));
    res = static_cast<P>(v);
    return AKM_SUCCESS;
  }

  //! A new cycle: |x|^2 partials of x; the steps' numbers follow the start's.
  int sumsq(const P *x)
  {
    if (seq != nullptr)
    {
      // past every number the cycle before may still publish
      start_seq = *seq + 1;
      *seq = start_seq + restart + 1;
    }
    finished = -2;
    gm_sumsq<P><<<ndot, gm_threads, 0, s>>>(n, drows, x, sqp);
    return check_launch("gmres norm");
  }

  //! |x| of a vector that is only read.
  int norm(const P *x, P &out)
  {
    AKM_TRY(sumsq(x));
    AKM_TRY(finish_step(-1, P{0}));
    return wait_step(-1, out);
  }

  //! V_0 holds a residual r: g_0 = |r| and 1/|r| beside it, finished by the
  //! first step's dot products (or finish_start).
  int start_async()
  {
    AKM_TRY(sumsq(V));
    if (lazy)
      return AKM_SUCCESS;
    AKM_TRY(finish_step(-1, P{0}));
    gm_scale<P><<<sblocks, gm_threads, 0, s>>>(n, V, st);
    return check_launch("gmres restart");
  }
  //! start_async, then beta = |r|.
  int start(P &beta)
  {
    AKM_TRY(start_async());
    if (finished < -1)
      AKM_TRY(finish_step(-1, P{0}));
    return wait_step(-1, beta);
  }

  //! Enqueues Arnoldi step j: z_j = pre(v_j) (flexible) or v_j, w = op(z_j),
  //! CGS against V_0..V_j, and beside it what is left of the step before.
  int launch_step(int j, std::function<int(const P *, P *)> const &op,
                  std::function<int(const P *, P *)> const *pre, P tol)
  {
    const P *vj = V + int64_t(j) * ldv;
    P *w = V + int64_t(j + 1) * ldv;
    const P *zj = vj;
    if (pre != nullptr)
    {
      P *zz = Z + int64_t(j) * ldv;
      AKM_TRY((*pre)(vj, zz));
      zj = zz;
    }
    AKM_TRY(op(zj, w));
    const int ncols = j + 1;
    const int extra = (finished < j - 1) ? 1 : 0;
    const dim3 grid(ndot + extra, (ncols + gm_cols - 1) / gm_cols);
    gm_dots<P><<<grid, gm_threads, extra * 3 * sizeof(P) * j, s>>>(
        n, drows, V, ldv, w, ncols, ndot, dotp, arrays(), pending(j - 1, tol));
    finished = std::max(finished, j - 1);
    gm_update<P><<<nupd, gm_upd_threads, sizeof(P) * ncols, s>>>(n, urows, V, ldv, w, j, dotp,
                                                                 ndot, arrays());
    if (!lazy)
    {
      AKM_TRY(finish_step(j, tol));
      gm_scale<P><<<sblocks, gm_threads, 0, s>>>(n, w, st);
    }
    return check_launch("gmres inner iteration");
  }

  //! Arnoldi steps 0, 1, ... until the estimate reaches `stop` or `limit`
  //! steps ran; count = the steps taken.  With `speculate`, step j + 1 is
  //! enqueued before step j's estimate is read (it finishes step j), which
  //! keeps the GPU busy through the host's round trips.  When step j ends the
  //! cycle the speculative step's columns, Hessenberg columns, rotations and
  //! g entries are never used (the update reads columns and g entries below
  //! count only), and the stream runs them before any later work.  With
  //! `beta_pending` the first steps also go out before the start's norm is
  //! known; when that norm already meets `stop` they are never used (count 0).
  int run_steps(int limit, std::function<int(const P *, P *)> const &op,
                std::function<int(const P *, P *)> const *pre, P tol, P stop, P &est,
                int &count, bool speculate, bool beta_pending = false)
  {
    // the start and the steps in flight each have a host slot of their own
    static_assert(gm_ahead + 2 <= gm_slots, "steps in flight exceed the state slots");
    // without slots the host copies the device state: one step at a time
    const int depth = (speculate && slots != nullptr) ? gm_ahead + 1 : 1;
    count = 0;
    int launched = 0;
    if (beta_pending)
    {
      while (launched < depth && launched < limit)
        AKM_TRY(launch_step(launched++, op, pre, tol));
      AKM_TRY(wait_step(-1, est));
    }
    while (est > stop && count < limit)
    {
      while (launched < count + depth && launched < limit)
        AKM_TRY(launch_step(launched++, op, pre, tol));
      if (finished < count)
        AKM_TRY(finish_step(count, tol));
      AKM_TRY(wait_step(count, est));
      ++count;
    }
    return AKM_SUCCESS;
  }

  //! x += B[:, 0:m] H^-1 g with B = Z (flexible) or V.
  int finish(int m, P *x, bool flexible)
  {
    if (m <= 0)
      return AKM_SUCCESS;
    const P *norms = (lazy && !flexible) ? inv : nullptr;
    if (m <= wave_size)
      gm_backsolve_wave<P><<<1, wave_size, 0, s>>>(m, H, g, norms);
    else
    {
      const size_t hbytes = sizeof(P) * (size_t(m) * (m + 1) / 2);
      const int h_in_lds = (hbytes + sizeof(P) * m <= 48 * 1024) ? 1 : 0;
      gm_backsolve<P><<<1, 256, sizeof(P) * m + (h_in_lds ? hbytes : 0), s>>>(m, H, g, h_in_lds,
                                                                             norms);
    }
    gm_xupdate<P><<<nupd, gm_upd_threads, sizeof(P) * m, s>>>(n, urows, flexible ? Z : V, ldv, m,
                                                              g, x);
    return check_launch("gmres update");
  }
};

//! The restart loop of simple_gmres (src/solver.cpp:201-295) on a cycle:
//! `residual(outer, speculate)` writes b - op(x) (preconditioned, for a left
//! preconditioner) into V_0 and may set `speculate`; then the Arnoldi steps,
//! the update of x and the absolute test of the residual estimate.
template<typename P, typename R>
static int gmres_outer(gm_cycle<P> &cyc, R &&residual,
                       std::function<int(const P *, P *)> const &op, P *x, int restart,
                       int max_outer, P tol, double *err, int *iterations)
{
  int total = 0, outer = 0;
  P inner_res = 0, outer_res = tol + 1;
  bool speculate = false;
  while (outer_res > tol && outer < max_outer)
  {
    AKM_TRY(residual(outer, speculate));
    ++total;
    // with host slots the host reads the start's norm only once the first
    // steps are enqueued
    const bool pending = cyc.slots != nullptr;
    if (pending)
      AKM_TRY(cyc.start_async());
    else
      AKM_TRY(cyc.start(inner_res));
    int inner = 0;
    AKM_TRY(cyc.run_steps(restart, op, nullptr, tol, tol, inner_res, inner, speculate, pending));
    total += inner;
    AKM_TRY(cyc.finish(inner, x, false));
    ++outer;
    outer_res = inner_res;
  }
  AKM_HIP(hipStreamSynchronize(cyc.s));
  if (err)
    *err = static_cast<double>(outer_res);
  if (iterations)
    *iterations = total;
  return (outer_res > tol) ? AKM_ERR_NOT_CONVERGED : AKM_SUCCESS;
}

//! The solve of akm_gmres_euler on device vectors in the memory `mem`.
//! Without host slots in `mem` the host waits for the whole stream after
//! every step, and no step is enqueued ahead.
template<typename P>
static int gmres_typed(akm_matrix_s &m, gm_memory const &mem, P dt, P *x, const P *b,
                       int restart, int max_outer, P tol, double *err, int *iterations)
{
  const int64_t n = m.output_size();
  hipStream_t s = m.stream;
  gm_cycle<P> cyc(mem, n, s, restart, nullptr, 0);
  P *V = cyc.V;
  // the global operator's solve is left-preconditioned by its Jacobi
  // diagonal, fused into the apply (src/solver.cpp:94-118)
  const bool jacobi = (m.mode == mode_global);
  auto apply_op = [&](P alpha, const P *v, P beta, P *w, P gamma, const P *g) -> int {
    if (jacobi)
      return global_apply(m, alpha, v, beta, w, gamma, g, true, static_cast<double>(dt));
    return apply_device(m, alpha, v, beta, w, gamma, g);
  };
  const std::function<int(const P *, P *)> op = [&](const P *v, P *w) -> int {
    return apply_op(-dt, v, P{0}, w, P{1}, v);
  };
  // r = b - (I - dt A) x into V_0; the first one is timed (when steps may be
  // in flight) to decide whether steps are enqueued ahead
  auto residual = [&](int outer, bool &speculate) -> int {
    AKM_HIP(hipMemcpyAsync(V, b, sizeof(P) * n, hipMemcpyDeviceToDevice, s));
    if (outer == 0 && mem.slots != nullptr)
    {
      // the first solve on the handle times its first apply (a host wait);
      // later solves reuse that time
      if (m.gmres_apply_ms < 0)
      {
        double ms = 0;
        AKM_TRY(timed_on_stream(
            s, [&]() { return apply_op(-dt * P{-1}, x, P{1}, V, P{-1}, x); }, ms));
        m.gmres_apply_ms = ms;
        speculate = ms < speculate_below_ms;
        return AKM_SUCCESS;
      }
      speculate = m.gmres_apply_ms < speculate_below_ms;
    }
    return apply_op(-dt * P{-1}, x, P{1}, V, P{-1}, x);
  };
  return gmres_outer<P>(cyc, residual, op, x, restart, max_outer, tol, err, iterations);
}

//! The mixed-precision / flexible solver (FP64 matrix m64).
static int gmres_mixed(akm_matrix_s &m64, akm_matrix_s *m32, akm_precond_s *pre, double dt,
                       double *x, const double *b, int restart, int max_cycles, double tol_rel,
                       double inner_rel, akm_solve_stats &stats)
{
  const int64_t n = m64.output_size();
  hipStream_t s = m64.stream;
  auto &ws = *m64.gmres;
  double *Z = (pre != nullptr) ? ws.Z.data() : nullptr;
  gm_cycle<double> cyc(memory_of(ws), n, s, restart, Z, 1);
  // a preconditioner may be nonlinear: it reads unit vectors
  cyc.lazy = pre == nullptr;
  double *V = cyc.V;
  const int sblocks = cyc.sblocks;

  std::function<int(const double *, double *)> op64 = [&](const double *v, double *w) -> int {
    ++stats.applies_f64;
    return apply_device(m64, -dt, v, 0.0, w, 1.0, v);
  };
  double bnorm = 0, beta = 0; // |b|, and |r| of the current cycle
  std::function<int(const double *, double *)> op32 = [&](const double *v, double *w) -> int {
    ++stats.applies_f32;
    // V_0 is the residual itself, at the scale of b, as the guess is taken to
    // be; the other vectors of a cycle have the norms of their steps
    const double scale = (v == x) ? f32_scale(bnorm)
                                  : ((cyc.lazy && v == V) ? f32_scale(beta) : 1.0);
    if (scale == 1.0 && apply_f32_between(*m32, v, -dt, w))
      return check_launch("gmres fp32 apply");
    gm_to_f32<<<sblocks, gm_threads, 0, s>>>(n, v, scale, ws.v32.data());
    AKM_TRY(check_launch("gmres fp32 cast"));
    AKM_TRY(apply_device(*m32, 1.0, ws.v32.data(), 0.0, ws.y32.data(), 0.0, nullptr));
    gm_axpy_f32<<<sblocks, gm_threads, 0, s>>>(n, v, -dt / scale, ws.y32.data(), w);
    return check_launch("gmres fp32 axpy");
  };
  std::function<int(const double *, double *)> precond = [&](const double *v,
                                                             double *z) -> int {
    ++stats.precond_applies;
    return pre->apply(v, z, s);
  };
  // r = b - (I - dt A) x in FP64 into V_0; norm = |r|
  auto true_residual = [&](double &norm) -> int {
    AKM_HIP(hipMemcpyAsync(V, b, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    ++stats.applies_f64;
    AKM_TRY(apply_device(m64, dt, x, 1.0, V, -1.0, x));
    return cyc.start(norm);
  };

  AKM_TRY(cyc.norm(b, bnorm));
  stats.rhs_norm = bnorm;
  if (bnorm == 0.0)
  {
    // the solution of (I - dt A) x = 0 is x = 0
    AKM_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, s));
    AKM_HIP(hipStreamSynchronize(s));
    stats.converged = 1;
    return AKM_SUCCESS;
  }
  const double tol_abs = tol_rel * bnorm;
  const auto &inner_op = (m32 != nullptr) ? op32 : op64;
  // with an FP32 operator a cycle cannot resolve the FP64 residual below
  // ~FP32 epsilon, so it stops at inner_rel of its starting residual
  const double cycle_rel = (m32 != nullptr) ? inner_rel : 0.0;

  double first_ms = 0;
  if (m32 != nullptr)
  {
    // the first cycle only needs its residual to the accuracy of its own
    // target (inner_rel of it): b - x in FP64 and dt*A*x with the FP32 operator
    AKM_TRY(timed_on_stream(s, [&]() { return op32(x, V); }, first_ms));
    gm_rsub<double><<<sblocks, gm_threads, 0, s>>>(n, b, V);
    AKM_TRY(check_launch("gmres residual"));
    AKM_TRY(cyc.start(beta));
  }
  else
  {
    AKM_HIP(hipMemcpyAsync(V, b, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    ++stats.applies_f64;
    AKM_TRY(timed_on_stream(s, [&]() { return apply_device(m64, dt, x, 1.0, V, -1.0, x); },
                            first_ms));
    AKM_TRY(cyc.start(beta));
  }
  // speculative steps pay off when a step's operator is cheap next to the
  // host round trip; the preconditioner (if any) runs in every step too
  const bool speculate = (pre == nullptr) && first_ms < speculate_below_ms;
  bool fallback = false;
  while (beta > tol_abs && stats.cycles < max_cycles)
  {
    const double stop = std::max(0.5 * tol_abs, cycle_rel * beta);
    if (!fallback)
      AKM_HIP(hipMemcpyAsync(ws.xprev.data(), x, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
    const auto &op = fallback ? op64 : inner_op;
    const auto *pc = (fallback || pre == nullptr) ? nullptr : &precond;
    double est = beta;
    int inner = 0;
    AKM_TRY(cyc.run_steps(restart, op, pc, stop, stop, est, inner, speculate && !fallback));
    AKM_TRY(cyc.finish(inner, x, pc != nullptr));
    stats.iterations += inner;
    if (fallback)
      stats.fallback_iterations += inner;
    ++stats.cycles;
    double beta_new = 0;
    AKM_TRY(true_residual(beta_new));
    if (!fallback && !(beta_new <= 0.5 * beta))
    {
      // the cycle did not halve the FP64 residual: undo it, go plain FP64
      AKM_HIP(hipMemcpyAsync(x, ws.xprev.data(), sizeof(double) * n, hipMemcpyDeviceToDevice, s));
      fallback = true;
      stats.fallback = 1;
      AKM_TRY(true_residual(beta));
      continue;
    }
    beta = beta_new;
  }
  AKM_HIP(hipStreamSynchronize(s));
  stats.abs_residual = beta;
  stats.rel_residual = beta / bnorm;
  stats.converged = (beta <= tol_abs) ? 1 : 0;
  return stats.converged ? AKM_SUCCESS : AKM_ERR_NOT_CONVERGED;
}

//! default_gmres_restarts (src/solver.cpp:142-152): clamp(512 MB / size, min(10, n), min(200, n)).
static int default_restarts(int64_t n, size_t esize)
{
  const int minimum = static_cast<int>(std::min<int64_t>(10, n));
  const int maximum = static_cast<int>(std::min<int64_t>(200, n));
  const double mb = double(n) * double(esize) / (1024.0 * 1024.0);
  int guess = static_cast<int>(512.0 / mb);
  return std::clamp(guess, minimum, maximum);
}

//! Sizes the workspace for n unknowns, `restart` and elements of `esize`
//! bytes (no work when it already has that shape).
static int size_workspace(akm_gmres_workspace &ws, int64_t n, int restart, size_t esize)
{
  if (ws.restart == restart && ws.n == n && ws.esize == esize)
    return AKM_SUCCESS;
  ws.restart = restart;
  ws.n = n;
  ws.esize = esize;
  AKM_TRY(ws.V.allocate(n * (restart + 1) * int64_t(esize)));
  AKM_TRY(ws.work.allocate(gm_work_values(n, restart) * int64_t(esize)));
  AKM_TRY(ws.state.allocate(sizeof(gm_state<double>)));
  AKM_TRY(ws.xb.allocate(2 * n * int64_t(esize)));
  if (ws.host_state == nullptr)
  {
    // coherent: a running kernel's stores are seen by the polling host
    AKM_HIP(hipHostMalloc(reinterpret_cast<void **>(&ws.host_state),
                          gm_slots * sizeof(gm_host_state), hipHostMallocCoherent));
    for (int i = 0; i < gm_slots; i++)
      ws.host_state[i] = gm_host_state{};
  }
  // buffers of the flexible / mixed solver are sized on first use
  ws.Z.reset();
  ws.xprev.reset();
  ws.v32.reset();
  ws.y32.reset();
  return AKM_SUCCESS;
}

static int ensure_workspace(akm_matrix_s &m, int restart)
{
  if (!m.gmres)
    m.gmres = std::unique_ptr<akm_gmres_workspace, void (*)(akm_gmres_workspace *)>(
        new akm_gmres_workspace(), delete_workspace);
  return size_workspace(*m.gmres, m.output_size(), restart, m.esize);
}

//! LU factorisation with partial pivoting of the n x n column-major a, in
//! place (getrf): piv[k] is the row swapped with row k at step k.  Returns
//! false for an exactly singular matrix.
template<typename P>
static bool lu_factor(int n, std::vector<P> &a, std::vector<int> &piv)
{
  piv.assign(n, 0);
  for (int k = 0; k < n; k++)
  {
    int p = k;
    for (int i = k + 1; i < n; i++)
      if (std::abs(a[int64_t(k) * n + i]) > std::abs(a[int64_t(k) * n + p]))
        p = i;
    piv[k] = p;
    if (a[int64_t(k) * n + p] == P{0})
      return false;
    if (p != k)
      for (int j = 0; j < n; j++)
        std::swap(a[int64_t(j) * n + k], a[int64_t(j) * n + p]);
    const P inv = P{1} / a[int64_t(k) * n + k];
    for (int i = k + 1; i < n; i++)
      a[int64_t(k) * n + i] *= inv;
    for (int j = k + 1; j < n; j++)
    {
      const P akj = a[int64_t(j) * n + k];
      if (akj != P{0})
        for (int i = k + 1; i < n; i++)
          a[int64_t(j) * n + i] -= a[int64_t(k) * n + i] * akj;
    }
  }
  return true;
}

//! simple_gmres on an explicit matrix (src/solver.cpp:54-74): host A, x, b
//! and optional M; the solve on the null stream with its own workspace.
template<typename P>
static int gmres_dense_typed(int n, const P *A_h, P *x_h, const P *b_h, const P *M_h,
                             int restart, int max_outer, P tol, double *err, int *iterations)
{
  constexpr int max_lu = 4096; // v in one workgroup's LDS
  if (M_h != nullptr && n > max_lu)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres dense: preconditioner of order %d above %d", n,
                     max_lu);
  hipStream_t s = nullptr;
  dev_buffer<P> A, xb, LU;
  dev_buffer<int> piv;
  AKM_TRY(A.upload(A_h, int64_t(n) * n, s));
  AKM_TRY(xb.allocate(2 * int64_t(n)));
  P *x = xb.data();
  P *b = xb.data() + n;
  AKM_HIP(hipMemcpyAsync(x, x_h, sizeof(P) * n, hipMemcpyHostToDevice, s));
  AKM_HIP(hipMemcpyAsync(b, b_h, sizeof(P) * n, hipMemcpyHostToDevice, s));
  if (M_h != nullptr)
  {
    std::vector<P> lu(M_h, M_h + int64_t(n) * n);
    std::vector<int> p;
    if (!lu_factor<P>(n, lu, p))
      return set_error(AKM_ERR_INVALID, "gmres dense: the preconditioner is singular");
    AKM_TRY(LU.upload(lu.data(), int64_t(n) * n, s));
    AKM_TRY(piv.upload(p.data(), n, s));
  }
  akm_gmres_workspace ws;
  AKM_TRY(size_workspace(ws, n, restart, sizeof(P)));
  gm_cycle<P> cyc(memory_of(ws), n, s, restart, nullptr, 0);
  const int gblocks = (n + gm_threads - 1) / gm_threads;
  auto precondition = [&](P *v) -> int {
    if (M_h == nullptr)
      return AKM_SUCCESS;
    gm_lu_solve<P><<<1, 256, sizeof(P) * n, s>>>(n, LU.data(), piv.data(), v);
    return check_launch("gmres dense preconditioner");
  };
  const std::function<int(const P *, P *)> op = [&](const P *v, P *w) -> int {
    gm_dense_gemv<P><<<gblocks, gm_threads, 0, s>>>(n, A.data(), v, P{1}, P{0}, w);
    AKM_TRY(check_launch("gmres dense gemv"));
    return precondition(w);
  };
  auto residual = [&](int, bool &) -> int {
    AKM_HIP(hipMemcpyAsync(cyc.V, b, sizeof(P) * n, hipMemcpyDeviceToDevice, s));
    gm_dense_gemv<P><<<gblocks, gm_threads, 0, s>>>(n, A.data(), x, P{-1}, P{1}, cyc.V);
    AKM_TRY(check_launch("gmres dense gemv"));
    return precondition(cyc.V);
  };
  const int rc = gmres_outer<P>(cyc, residual, op, x, restart, max_outer, tol, err, iterations);
  if (rc < 0)
    return rc;
  AKM_HIP(hipMemcpy(x_h, x, sizeof(P) * n, hipMemcpyDeviceToHost));
  return rc;
}


} // namespace akm

using namespace akm;

extern "C" akm_status akm_gmres_euler(akm_matrix mat, double dt, void *x, const void *b,
                                      int restart, int max_iter, double tol, int on_device,
                                      double *err, int *iterations)
{
  if (mat == nullptr || x == nullptr || b == nullptr)
    return set_error(AKM_ERR_INVALID, "gmres: null argument");
  if (mat->rows != mat->cols)
    return set_error(AKM_ERR_INVALID, "gmres: the operator must be square");
  const int64_t n = mat->output_size();
  if (n <= 0)
    return set_error(AKM_ERR_INVALID, "gmres: empty system");
  if (tol <= 0)
    tol = (mat->prec == AKM_F64) ? 1e-12 : 1e-6;
  if (restart <= 0)
    restart = default_restarts(n, mat->esize);
  if (restart > n)
    return set_error(AKM_ERR_INVALID, "Number of inner iterations %d must be less than %lld!",
                     restart, static_cast<long long>(n));
  if (restart > gm_max_restart)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres: restart %d above %d", restart, gm_max_restart);
  if (max_iter <= 0)
    max_iter = static_cast<int>(std::min<int64_t>(n, 1 << 30));
  AKM_TRY(ensure_workspace(*mat, restart));
  void *xd = x;
  const void *bd = b;
  auto &ws = *mat->gmres;
  const size_t bytes = size_t(n) * mat->esize;
  if (!on_device)
  {
    xd = ws.xb.data();
    bd = ws.xb.data() + bytes;
    AKM_HIP(hipMemcpyAsync(xd, x, bytes, hipMemcpyHostToDevice, mat->stream));
    AKM_HIP(hipMemcpyAsync(const_cast<void *>(bd), b, bytes, hipMemcpyHostToDevice,
                           mat->stream));
  }
  int rc;
  const gm_memory mem = memory_of(ws);
  if (mat->prec == AKM_F64)
    rc = gmres_typed<double>(*mat, mem, dt, static_cast<double *>(xd),
                             static_cast<const double *>(bd), restart, max_iter, tol, err,
                             iterations);
  else
    rc = gmres_typed<float>(*mat, mem, static_cast<float>(dt), static_cast<float *>(xd),
                            static_cast<const float *>(bd), restart, max_iter,
                            static_cast<float>(tol), err, iterations);
  if (rc < 0)
    return rc;
  if (!on_device)
  {
    AKM_HIP(hipMemcpyAsync(x, xd, bytes, hipMemcpyDeviceToHost, mat->stream));
    AKM_HIP(hipStreamSynchronize(mat->stream));
  }
  return rc;
}

// ------------------------------------------------- allocation-free solve ---

namespace akm
{
//! Device memory of akm_gmres_euler_noalloc: the Krylov basis, the small
//! work array and the step state of one solve.  Every GPU the library runs on
//! holds its own copy until the process ends.  Host code never passes this
//! name to a kernel or a copy: it resolves the array's device address once
//! per GPU (noalloc_memory) and uses that.
static __device__ __align__(256) unsigned char scratch[AKM_NOALLOC_SCRATCH_BYTES];

constexpr int noalloc_max_devices = 64;

//! Per GPU: the device address of `scratch` and the host copies of the step
//! state (plain host memory: the host waits for the stream before reading).
struct noalloc_slot
{
  void *dev = nullptr;
  alignas(64) unsigned char host[sizeof(gm_state<double>)];
};
static noalloc_slot noalloc_slots[noalloc_max_devices];
static std::mutex noalloc_mtx;

static int64_t round_up_256(int64_t b) { return (b + 255) / 256 * 256; }

//! Scratch bytes of a solve of n unknowns with `restart` of `esize` bytes.
static int64_t noalloc_bytes(int64_t n, int restart, size_t esize)
{
  return round_up_256(n * (restart + 1) * int64_t(esize)) +
         round_up_256(gm_work_values(n, restart) * int64_t(esize)) +
         round_up_256(int64_t(sizeof(gm_state<double>)));
}

//! The solve's memory carved from the current GPU's scratch array, resolving
//! its address on the first call on that GPU.  No host slots: the host waits for
//! the whole stream after every step and no step is enqueued ahead.
static int noalloc_memory(int64_t n, int restart, size_t esize, gm_memory &mem)
{
  int dev = 0;
  AKM_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= noalloc_max_devices)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres noalloc: device %d above %d", dev,
                     noalloc_max_devices - 1);
  noalloc_slot &slot = noalloc_slots[dev];
  {
    std::lock_guard<std::mutex> lock(noalloc_mtx);
    if (slot.dev == nullptr)
    {
      void *p = nullptr;
      AKM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      if (p == nullptr)
        return set_error(AKM_ERR_HIP, "gmres noalloc: no device address for the scratch array");
      slot.dev = p;
    }
  }
  unsigned char *base = static_cast<unsigned char *>(slot.dev);
  const int64_t vbytes = round_up_256(n * (restart + 1) * int64_t(esize));
  const int64_t wbytes = round_up_256(gm_work_values(n, restart) * int64_t(esize));
  mem.V = base;
  mem.work = base + vbytes;
  mem.state = base + vbytes + wbytes;
  mem.host_state = slot.host;
  return AKM_SUCCESS;
}
} // namespace akm

extern "C" akm_status akm_gmres_euler_noalloc(akm_matrix mat, double dt, void *x, const void *b,
                                              int restart, int max_iter, double tol, double *err,
                                              int *iterations)
{
  if (mat == nullptr || x == nullptr || b == nullptr)
    return set_error(AKM_ERR_INVALID, "gmres noalloc: null argument");
  if (mat->rows != mat->cols)
    return set_error(AKM_ERR_INVALID, "gmres noalloc: the operator must be square");
  const int64_t n = mat->output_size();
  if (n <= 0)
    return set_error(AKM_ERR_INVALID, "gmres noalloc: empty system");
  const int64_t cap = AKM_NOALLOC_SCRATCH_BYTES;
  if (tol <= 0)
    tol = (mat->prec == AKM_F64) ? 1e-12 : 1e-6;
  if (restart <= 0)
  {
    // the reference default, lowered until the basis fits the scratch array
    restart = default_restarts(n, mat->esize);
    while (restart > 1 && noalloc_bytes(n, restart, mat->esize) > cap)
      --restart;
  }
  if (restart > n)
    return set_error(AKM_ERR_INVALID, "Number of inner iterations %d must be less than %lld!",
                     restart, static_cast<long long>(n));
  if (restart > gm_max_restart)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres: restart %d above %d", restart, gm_max_restart);
  const int64_t need = noalloc_bytes(n, restart, mat->esize);
  if (need > cap)
    return set_error(AKM_ERR_INVALID,
                     "gmres noalloc: %lld unknowns with restart %d need %lld bytes of scratch, "
                     "above the fixed %lld",
                     static_cast<long long>(n), restart, static_cast<long long>(need),
                     static_cast<long long>(cap));
  if (max_iter <= 0)
    max_iter = static_cast<int>(std::min<int64_t>(n, 1 << 30));
  gm_memory mem;
  AKM_TRY(noalloc_memory(n, restart, mat->esize, mem));
  if (mat->prec == AKM_F64)
    return gmres_typed<double>(*mat, mem, dt, static_cast<double *>(x),
                               static_cast<const double *>(b), restart, max_iter, tol, err,
                               iterations);
  return gmres_typed<float>(*mat, mem, static_cast<float>(dt), static_cast<float *>(x),
                            static_cast<const float *>(b), restart, max_iter,
                            static_cast<float>(tol), err, iterations);
}

extern "C" akm_status akm_gmres_euler_mixed(akm_matrix mat, akm_matrix mat32, akm_precond pre,
                                            double dt, double *x, const double *b, int restart,
                                            int max_cycles, double tol, double inner_tol,
                                            akm_solve_stats *stats)
{
  if (mat == nullptr || x == nullptr || b == nullptr)
    return set_error(AKM_ERR_INVALID, "gmres: null argument");
  if (mat->prec != AKM_F64)
    return set_error(AKM_ERR_INVALID, "gmres mixed: the operator must be FP64");
  if (mat->rows != mat->cols)
    return set_error(AKM_ERR_INVALID, "gmres: the operator must be square");
  const int64_t n = mat->output_size();
  if (n <= 0)
    return set_error(AKM_ERR_INVALID, "gmres: empty system");
  if (mat32 != nullptr &&
      (mat32->prec != AKM_F32 || mat32->output_size() != n || mat32->input_size() != n))
    return set_error(AKM_ERR_INVALID,
                     "gmres mixed: the inner operator must be FP32 and of the same size");
  if (pre != nullptr && pre->size() != n)
    return set_error(AKM_ERR_INVALID, "gmres mixed: preconditioner size %lld != system size %lld",
                     static_cast<long long>(pre->size()), static_cast<long long>(n));
  if (tol <= 0)
    tol = 1e-10;
  if (inner_tol <= 0)
    inner_tol = 1e-6;
  if (restart <= 0)
    restart = default_restarts(n, mat->esize);
  if (restart > n)
    return set_error(AKM_ERR_INVALID, "Number of inner iterations %d must be less than %lld!",
                     restart, static_cast<long long>(n));
  if (restart > gm_max_restart)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres: restart %d above %d", restart, gm_max_restart);
  if (max_cycles <= 0)
    max_cycles = static_cast<int>(std::min<int64_t>(n, 1 << 30));
  AKM_TRY(ensure_workspace(*mat, restart));
  auto &ws = *mat->gmres;
  if (pre != nullptr && ws.Z.size() != n * restart)
    AKM_TRY(ws.Z.allocate(n * restart));
  AKM_TRY(ws.xprev.allocate(n));
  if (mat32 != nullptr)
  {
    AKM_TRY(ws.v32.allocate(n));
    AKM_TRY(ws.y32.allocate(n));
  }
  akm_solve_stats local{};
  hipStream_t saved = nullptr;
  if (mat32 != nullptr)
  {
    saved = mat32->stream;
    use_stream(*mat32, mat->stream); // one stream for the whole solve
  }
  int rc = gmres_mixed(*mat, mat32, pre, dt, x, b, restart, max_cycles, tol, inner_tol, local);
  if (mat32 != nullptr)
    use_stream(*mat32, saved);
  if (stats != nullptr)
    *stats = local;
  return rc;
}

extern "C" akm_status akm_gmres_dense(int n, const void *A, void *x, const void *b,
                                      const void *M, int restart, int max_iter, double tol,
                                      akm_prec prec, double *err, int *iterations)
{
  if (A == nullptr || x == nullptr || b == nullptr)
    return set_error(AKM_ERR_INVALID, "gmres dense: null argument");
  if (n <= 0)
    return set_error(AKM_ERR_INVALID, "gmres dense: empty system");
  if (prec != AKM_F64 && prec != AKM_F32)
    return set_error(AKM_ERR_INVALID, "gmres dense: unknown precision %d", int(prec));
  const size_t esize = (prec == AKM_F64) ? sizeof(double) : sizeof(float);
  if (tol <= 0)
    tol = (prec == AKM_F64) ? 1e-12 : 1e-6;
  if (restart <= 0)
    restart = default_restarts(n, esize);
  if (restart > n)
    return set_error(AKM_ERR_INVALID, "Number of inner iterations %d must be less than %d!",
                     restart, n);
  if (restart > gm_max_restart)
    return set_error(AKM_ERR_UNSUPPORTED, "gmres: restart %d above %d", restart, gm_max_restart);
  if (max_iter <= 0)
    max_iter = n;
  if (prec == AKM_F64)
    return gmres_dense_typed<double>(n, static_cast<const double *>(A), static_cast<double *>(x),
                                     static_cast<const double *>(b),
                                     static_cast<const double *>(M), restart, max_iter, tol,
                                     err, iterations);
  return gmres_dense_typed<float>(n, static_cast<const float *>(A), static_cast<float *>(x),
                                  static_cast<const float *>(b), static_cast<const float *>(M),
                                  restart, max_iter, static_cast<float>(tol), err, iterations);
}
