// Batched implicit-step solves: many independent systems
// (I - dt_s A_s) x_s = b_s, of any sizes and (d, n), iterate restarted GMRES
// in lockstep on the GPU.
//
// * Operators that run one dimension at a time in one stage (fibre.hip) are
//   applied together, one launch per workgroup size with a workgroup per
//   (system, group of slots).  The others are applied pair by pair, by a
//   persistent kernel per (d, n) group that walks a (system, row) work list
//   sorted longest row first across all the group's systems.
// * Every vector kernel runs over a global list of row blocks covering all
//   systems; per-system scalars (Hessenberg column, rotations, right-hand
//   side, norms) live in device arrays, and a system that converges or runs
//   out of its cycle is masked out by a device flag.  As in the single solver
//   (gmres.hip) a step is the apply, the dot products and the update; what
//   remains of a step (norm, rotation, estimate) is done by one extra
//   workgroup per system of the next step's dot products, and Krylov vectors
//   keep their 1/norm aside.
// * A restart cycle is three stream captures replayed as hipGraphs: the cycle
//   start (b - (I - dt A) x for every unconverged system, its norm and the
//   convergence test), bt_chunk Arnoldi iterations (columns *jcol .. *jcol +
//   bt_chunk - 1 below the restart; the graph advances the device counter
//   itself), and the update x += V H^-1 g.  The host reads the per-system
//   flags after every replay to stop early.
// * No memset is recorded in the graphs; all initialisation is by kernels.
//
// The arithmetic per system is the reference GMRES (src/solver.cpp:156-298)
// with classical Gram-Schmidt and Givens rotations, the residual estimate
// tested against tol*|b_s|, and the true residual recomputed at every cycle
// start (a system is converged when that true residual is below tolerance).
#include "fibre.hpp"
#include "matrix.hpp"

#include <algorithm>
#include <map>
#include <memory>
#include <numeric>
#include <vector>

namespace akm
{
//! Arnoldi iterations between two host reads of the batch state.
constexpr int bt_chunk = 8;

constexpr int bt_threads = 256;
constexpr int bt_cols = 4;   // Krylov columns per dot-product block
constexpr int bt_split = 4;  // threads that share a row's columns in the update
constexpr int bt_tile = 128; // rows of an update block at a time
constexpr int bt_upd_threads = bt_split * bt_tile;
constexpr int bt_lanes = 8;  // lanes that add one column's dot partials
constexpr int bt_max_restart = 255;

//! Static per-system data of the vector kernels.
struct bt_sys
{
  double *V;       // Krylov basis, (restart + 1) columns of n
  double *X;       // solution
  double *B;       // right-hand side
  int64_t n;
  int64_t drows, urows; // rows of a dot-product / update block
  int ndot, nupd;       // such blocks of this system
  int dot0, upd0;       // its first block in the global lists
  // Hessenberg column and packed columns, rotations, right-hand side, 1/norms
  // of the stored Krylov vectors, dot and |w|^2 partials
  double *h, *H, *cs, *sn, *g, *inv, *dotp, *sqp;
};

//! Mutable per-system state.
struct bt_state
{
  double tol; // absolute tolerance tol_rel * |b|
  double res; // residual estimate / true residual at cycle start
  int converged;
  int m;        // Krylov columns of the current cycle
  int iters;    // operator applications
  int finished; // last finished step of the cycle (-1: its start, -2: none)
  int open;     // the active flag, for the host
  int pad;
};

//! The caller's vectors of systems first .. first + count, by value.
constexpr int bt_vectors = 64;
struct bt_io
{
  double *x[bt_vectors];
  const double *b[bt_vectors];
  int first;
};

//! Fixed-order sum over the workgroup: a shuffle tree inside each wavefront,
//! then the wavefronts' sums in order.
__device__ __forceinline__ double bt_block_sum(double v, double *sh)
{
#pragma unroll
  for (int off = wave_size / 2; off > 0; off >>= 1)
    v += __shfl_xor(v, off, wave_size);
  if (threadIdx.x % wave_size == 0)
    sh[threadIdx.x / wave_size] = v;
  __syncthreads();
  double r = 0;
  for (int w = 0; w < static_cast<int>(blockDim.x) / wave_size; w++)
    r += sh[w];
  __syncthreads();
  return r;
}

//! Start of a cycle: active = open = !converged, m = 0; column counter = 0.
__global__ void bt_begin(int nsys, bt_state *st, int *active, int *open, int *jcol)
{
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s == 0)
    *jcol = 0;
  if (s < nsys)
  {
    const int on = st[s].converged ? 0 : 1;
    active[s] = open[s] = on;
    st[s].open = on;
    st[s].m = 0;
    st[s].finished = -2;
  }
}

//! V_s[0] = b_s for the active systems.
__global__ void __launch_bounds__(bt_threads)
bt_copy_rhs(const int *dot_sys, const bt_sys *sys, const int *active)
{
  const int s = dot_sys[blockIdx.x];
  if (!active[s])
    return;
  const bt_sys q = sys[s];
  const int64_t r0 = int64_t(blockIdx.x - q.dot0) * q.drows, r1 = min(q.n, r0 + q.drows);
  for (int64_t i = r0 + threadIdx.x; i < r1; i += bt_threads)
    q.V[i] = q.B[i];
}

//! X_s = x_s, B_s = b_s and the partials of |b_s|^2, all systems of `io` in
//! one launch (a copy per vector costs the host 4 us and the GPU 2).
__global__ void __launch_bounds__(bt_threads)
bt_load(const int *dot_sys, int block0, const bt_sys *sys, bt_io io)
{
  __shared__ double sh[bt_threads / wave_size];
  const int s = dot_sys[block0 + blockIdx.x];
  const bt_sys q = sys[s];
  const int lb = block0 + blockIdx.x - q.dot0;
  const int64_t r0 = int64_t(lb) * q.drows, r1 = min(q.n, r0 + q.drows);
  const double *x = io.x[s - io.first], *b = io.b[s - io.first];
  double sq = 0;
  for (int64_t i = r0 + threadIdx.x; i < r1; i += bt_threads)
  {
    const double bi = b[i];
    q.X[i] = x[i];
    q.B[i] = bi;
    sq = fma(bi, bi, sq);
  }
  sq = bt_block_sum(sq, sh);
  if (threadIdx.x == 0)
    q.sqp[lb] = sq;
}

//! x_s = X_s.
__global__ void __launch_bounds__(bt_threads)
bt_store(const int *dot_sys, int block0, const bt_sys *sys, bt_io io)
{
  const int s = dot_sys[block0 + blockIdx.x];
  const bt_sys q = sys[s];
  const int64_t r0 = int64_t(block0 + blockIdx.x - q.dot0) * q.drows, r1 = min(q.n, r0 + q.drows);
  double *x = io.x[s - io.first];
  for (int64_t i = r0 + threadIdx.x; i < r1; i += bt_threads)
    x[i] = q.X[i];
}

//! sq partials of |V_s[0]|^2.
__global__ void __launch_bounds__(bt_threads)
bt_sumsq(const int *dot_sys, const bt_sys *sys, const int *active)
{
  __shared__ double sh[bt_threads / wave_size];
  const int s = dot_sys[blockIdx.x];
  if (!active[s])
    return;
  const bt_sys q = sys[s];
  const int lb = blockIdx.x - q.dot0;
  const int64_t r0 = int64_t(lb) * q.drows, r1 = min(q.n, r0 + q.drows);
  double sq = 0;
  for (int64_t i = r0 + threadIdx.x; i < r1; i += bt_threads)
    sq = fma(q.V[i], q.V[i], sq);
  sq = bt_block_sum(sq, sh);
  if (threadIdx.x == 0)
    q.sqp[lb] = sq;
}

//! Per system: tol = tol_rel * |b|, converged = 0, iters = 0.
__global__ void __launch_bounds__(64) bt_set_tol(const bt_sys *sys, bt_state *st, double tol_rel)
{
  __shared__ double sh[1];
  const int s = blockIdx.x;
  const bt_sys q = sys[s];
  double v = 0;
  for (int b = threadIdx.x; b < q.ndot; b += 64)
    v += q.sqp[b];
  v = bt_block_sum(v, sh);
  if (threadIdx.x == 0)
  {
    st[s].tol = tol_rel * sqrt(v);
    st[s].converged = 0;
    st[s].iters = 0;
    st[s].m = 0;
  }
}

__device__ __forceinline__ void bt_rot(double &x, double &y, double c, double s)
{
  const double t = c * x + s * y;
  y = c * y - s * x;
  x = t;
}

//! reference BLAS rotg semantics
__device__ __forceinline__ void bt_rotg(double &a, double b, double &c, double &s)
{
  const double roe = (fabs(a) > fabs(b)) ? a : b;
  const double scale = fabs(a) + fabs(b);
  if (scale == 0.0)
  {
    c = 1;
    s = 0;
    a = 0;
    return;
  }
  const double as = a / scale, bs = b / scale;
  double r = scale * sqrt(as * as + bs * bs);
  r = (roe >= 0.0) ? r : -r;
  c = a / r;
  s = b / r;
  a = r;
}

//! One workgroup finishes step j of system s (j < 0: the cycle's start, with
//! the convergence test on the true residual): |w|, Hessenberg column j, old
//! rotations, the new one, the estimate; m = j + 1; a system whose estimate is
//! below tolerance leaves the cycle: open = 0.  `active` is only read: row
//! workgroups of the same launch read it too, and the update after them takes
//! it over from `open`.
__device__ __forceinline__ void bt_finish_step(bt_sys const &q, bt_state *st, const int *active,
                                               int *open, int s, int j)
{
  __shared__ double sh[bt_threads / wave_size];
  __shared__ double lc[bt_max_restart], lcs[bt_max_restart], lsn[bt_max_restart];
  const int t = threadIdx.x;
  if (!active[s] || st[s].finished >= j)
    return; // the same in every thread
  for (int k = t; k <= j; k += blockDim.x)
    lc[k] = q.h[k];
  for (int k = t; k < j; k += blockDim.x)
  {
    lcs[k] = q.cs[k];
    lsn[k] = q.sn[k];
  }
  double v = 0;
  for (int b = t; b < ((j < 0) ? q.ndot : q.nupd); b += blockDim.x)
    v += q.sqp[b];
  v = bt_block_sum(v, sh); // its barriers also order the reads above
  const double nrm = sqrt(v);
  if (t == 0)
  {
    bt_state &state = st[s];
    q.inv[j + 1] = (nrm > 0.0) ? 1.0 / nrm : 0.0;
    state.iters += 1;
    state.finished = j;
    if (j < 0)
    {
      q.g[0] = nrm;
      state.res = nrm;
      if (nrm <= state.tol)
      {
        state.converged = 1;
        state.open = 0;
        open[s] = 0;
      }
    }
    else
    {
      // down the column, the running entry in a register
      double x = lc[0];
      for (int k = 0; k < j; k++)
      {
        double y = lc[k + 1];
        bt_rot(x, y, lcs[k], lsn[k]);
        lc[k] = x;
        x = y;
      }
      double c, sv;
      bt_rotg(x, nrm, c, sv);
      lc[j] = x;
      q.cs[j] = c;
      q.sn[j] = sv;
      double gj = q.g[j], gn = 0;
      bt_rot(gj, gn, c, sv);
      q.g[j] = gj;
      q.g[j + 1] = gn;
      state.res = fabs(gn);
      state.m = j + 1;
      if (state.res <= state.tol)
      {
        state.open = 0;
        open[s] = 0;
      }
    }
  }
  __syncthreads();
  for (int k = t; k <= j; k += blockDim.x)
    q.H[(j * (j + 1)) / 2 + k] = lc[k];
}

//! Finishes the start of the cycle (advance = 0), or the last step of a chunk
//! of `advance` iterations.
__global__ void __launch_bounds__(bt_threads)
bt_finish(const bt_sys *sys, bt_state *st, int *active, int *open, const int *jcol, int advance,
          int limit)
{
  const int s = blockIdx.x;
  bt_finish_step(sys[s], st, active, open, s,
                 (advance == 0) ? -1 : min(*jcol + advance, limit) - 1);
  __syncthreads(); // every thread has read the flag
  if (threadIdx.x == 0)
    active[s] = open[s];
}

//! partial dots of V_s[k], k <= j, with w = V_s[j+1]; the workgroups past the
//! row blocks finish step j - 1 of their system.  The reduction is gm_dots'.
__global__ void __launch_bounds__(bt_threads)
bt_dots(const int *dot_sys, int total, const bt_sys *sys, bt_state *st, const int *active,
        int *open, const int *jcol, int joff, int limit)
{
  static_assert(bt_cols == 4, "the exchange below halves four columns twice");
  __shared__ double sh[bt_threads / wave_size][bt_cols];
  const int j = *jcol + joff;
  if (j >= limit)
    return;
  if (static_cast<int>(blockIdx.x) >= total)
  {
    const int s = blockIdx.x - total;
    if (blockIdx.y == 0)
      bt_finish_step(sys[s], st, active, open, s, j - 1);
    return;
  }
  const int s = dot_sys[blockIdx.x];
  const int ncols = j + 1;
  const int k0 = blockIdx.y * bt_cols;
  // a system that leaves in this launch is still taken here; the update
  // skips it
  if (k0 >= ncols || !active[s])
    return;
  const bt_sys q = sys[s];
  const int lb = blockIdx.x - q.dot0;
  const int64_t r0 = int64_t(lb) * q.drows, r1 = min(q.n, r0 + q.drows);
  const double *w = q.V + int64_t(ncols) * q.n;
  double acc[bt_cols];
  const double *col[bt_cols];
#pragma unroll
  for (int c = 0; c < bt_cols; c++)
  {
    acc[c] = 0;
    col[c] = q.V + int64_t(min(k0 + c, ncols - 1)) * q.n;
  }
#pragma unroll 4
  for (int64_t i = r0 + threadIdx.x; i < r1; i += bt_threads)
  {
    const double wi = w[i];
#pragma unroll
    for (int c = 0; c < bt_cols; c++)
      acc[c] = fma(col[c][i], wi, acc[c]);
  }
  const int lane = threadIdx.x % wave_size;
  const bool up = (lane & 32) != 0, odd = (lane & 16) != 0;
  const double a0 = (up ? acc[2] : acc[0]) + __shfl_xor(up ? acc[0] : acc[2], 32, wave_size);
  const double a1 = (up ? acc[3] : acc[1]) + __shfl_xor(up ? acc[1] : acc[3], 32, wave_size);
  double v = (odd ? a1 : a0) + __shfl_xor(odd ? a0 : a1, 16, wave_size);
#pragma unroll
  for (int off = 8; off > 0; off >>= 1)
    v += __shfl_xor(v, off, wave_size);
  if ((lane & 15) == 0)
    sh[threadIdx.x / wave_size][(up ? 2 : 0) + (odd ? 1 : 0)] = v;
  __syncthreads();
  if (threadIdx.x < bt_cols && k0 + static_cast<int>(threadIdx.x) < ncols)
  {
    double sum = 0;
#pragma unroll
    for (int w2 = 0; w2 < bt_threads / wave_size; w2++)
      sum += sh[w2][threadIdx.x];
    q.dotp[int64_t(k0 + threadIdx.x) * q.ndot + lb] = sum;
  }
}

//! h_s, then w <- w / |v_j| - V_s[0..j] h_s and the partials of |w|^2 for the
//! systems still open; a system's first workgroup takes its flag over.
__global__ void __launch_bounds__(bt_upd_threads)
bt_update(const int *upd_sys, const bt_sys *sys, int *active, const int *open, const int *jcol,
          int joff, int limit)
{
  __shared__ double red[bt_split][bt_tile];
  __shared__ double sh[bt_upd_threads / wave_size];
  __shared__ double cf[bt_max_restart]; // h_k / |stored v_k|
  const int s = upd_sys[blockIdx.x];
  const int j = *jcol + joff;
  if (j >= limit)
    return;
  const bt_sys q = sys[s];
  const int t = threadIdx.x, ncols = j + 1, lb = blockIdx.x - q.upd0;
  const int on = open[s]; // not written in this launch
  if (lb == 0 && t == 0)
    active[s] = on;
  if (on == 0)
    return;
  const double invj = q.inv[j];
  for (int k = t / bt_lanes; k < ncols; k += bt_upd_threads / bt_lanes)
  {
    const double ik = q.inv[k];
    double v = 0;
#pragma unroll 8
    for (int b = t % bt_lanes; b < q.ndot; b += bt_lanes)
      v += q.dotp[int64_t(k) * q.ndot + b];
#pragma unroll
    for (int off = bt_lanes / 2; off > 0; off >>= 1)
      v += __shfl_xor(v, off, wave_size);
    if (t % bt_lanes == 0)
    {
      const double h = v * ik * invj;
      cf[k] = h * ik;
      if (lb == 0)
        q.h[k] = h;
    }
  }
  __syncthreads();
  const int part = t / bt_tile, lane = t % bt_tile;
  const int64_t r0 = int64_t(lb) * q.urows, r1 = min(q.n, r0 + q.urows);
  double *w = q.V + int64_t(ncols) * q.n;
  double sq = 0;
  for (int64_t base = r0; base < r1; base += bt_tile)
  {
    const int64_t i = base + lane;
    double acc = 0;
    if (i < r1)
    {
#pragma unroll 8
      for (int k = part; k < ncols; k += bt_split)
        acc = fma(q.V[int64_t(k) * q.n + i], cf[k], acc);
    }
    red[part][lane] = acc;
    __syncthreads();
    if (part == 0 && i < r1)
    {
      double sum = red[0][lane];
#pragma unroll
      for (int p = 1; p < bt_split; p++)
        sum += red[p][lane];
      const double v = fma(w[i], invj, -sum);
      w[i] = v;
      sq = fma(v, v, sq);
    }
    __syncthreads();
  }
  sq = bt_block_sum(sq, sh);
  if (t == 0)
    q.sqp[lb] = sq;
}

__global__ void bt_advance(int *jcol, int by)
{
  if (threadIdx.x == 0 && blockIdx.x == 0)
    *jcol += by;
}

//! y = H^-1 g (packed upper triangle), then y_k / |stored v_k|, for every
//! system with m > 0: a wavefront per system, the updates of a column over
//! the lanes.
__global__ void __launch_bounds__(64)
bt_backsolve(const bt_sys *sys, const bt_state *st)
{
  __shared__ double lg[bt_max_restart];
  const int s = blockIdx.x, lane = threadIdx.x;
  const int m = st[s].m;
  if (m <= 0)
    return;
  const bt_sys q = sys[s];
  for (int i = lane; i < m; i += 64)
    lg[i] = q.g[i];
  __syncthreads();
  for (int j = m - 1; j >= 0; j--)
  {
    const double *col = q.H + (j * (j + 1)) / 2;
    const double hjj = col[j];
    const double gj = (hjj != 0.0) ? lg[j] / hjj : 0.0;
    __syncthreads();
    for (int i = lane; i < j; i += 64)
      lg[i] -= gj * col[i];
    if (lane == 0)
      lg[j] = gj;
    __syncthreads();
  }
  for (int i = lane; i < m; i += 64)
    q.g[i] = lg[i] * q.inv[i];
}

//! x_s += V_s[0..m) y_s.
__global__ void __launch_bounds__(bt_upd_threads)
bt_xupdate(const int *upd_sys, const bt_sys *sys, const bt_state *st)
{
  __shared__ double red[bt_split][bt_tile];
  __shared__ double ys[bt_max_restart];
  const int s = upd_sys[blockIdx.x];
  const int m = st[s].m;
  if (m <= 0)
    return;
  const bt_sys q = sys[s];
  for (int k = threadIdx.x; k < m; k += bt_upd_threads)
    ys[k] = q.g[k];
  __syncthreads();
  const int part = threadIdx.x / bt_tile, lane = threadIdx.x % bt_tile;
  const int64_t r0 = int64_t(blockIdx.x - q.upd0) * q.urows, r1 = min(q.n, r0 + q.urows);
  for (int64_t base = r0; base < r1; base += bt_tile)
  {
    const int64_t i = base + lane;
    double acc = 0;
    if (i < r1)
    {
#pragma unroll 8
      for (int k = part; k < m; k += bt_split)
        acc = fma(q.V[int64_t(k) * q.n + i], ys[k], acc);
    }
    red[part][lane] = acc;
    __syncthreads();
    if (part == 0 && i < r1)
    {
      double sum = red[0][lane];
#pragma unroll
      for (int p = 1; p < bt_split; p++)
        sum += red[p][lane];
      q.X[i] += sum;
    }
    __syncthreads();
  }
}

//! dst = value on n entries (kernel fill: no memset nodes in the graphs).
__global__ void __launch_bounds__(bt_threads) bt_fill(int64_t n, double *dst, double value)
{
  for (int64_t i = blockIdx.x * int64_t(bt_threads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * bt_threads)
    dst[i] = value;
}

} // namespace akm

using namespace akm;

struct akm_batch_s
{
  //! Systems applied pair by pair, by (d, n).
  struct group
  {
    int d = 0, n = 0, waves = 4, grid = 1;
    dev_buffer<int2> work;
    int nwork = 0;
  };
  //! Systems applied along fibres, by workgroup size.
  struct walk
  {
    int tpb = 256, groups = 0;
    dev_buffer<int2> items;
  };
  int nsys = 0, restart = 0;
  int64_t total_n = 0;
  int dot_blocks = 0, upd_blocks = 0;
  std::vector<akm_matrix> mats;
  std::vector<uint64_t> forms;    // the matrices' form stamps the plans are for
  std::vector<fibre_plan> plans;  // per system (not built: pair by pair)
  std::vector<int64_t> n_of, x_off;
  std::vector<group> groups;
  std::vector<walk> walks;
  std::vector<int> waves_of_dn; // per (d, n): wavefronts per row, 1 for walks
  dev_buffer<kron_args<double>> args;
  dev_buffer<fibre_system> fsys;
  dev_buffer<batch_system> vsys;
  std::vector<batch_system> host_vsys;
  dev_buffer<bt_sys> sys;
  dev_buffer<bt_state> state;
  dev_buffer<int> active, open_dev, jcol, dot_sys, upd_sys;
  dev_buffer<double> V, X, B, small;
  bt_state *host_state = nullptr; // pinned
  std::vector<int> dot0;          // first dot-product block per system, and the total
  hipStream_t stream = nullptr; // own stream (the null stream cannot be captured)
  hipGraphExec_t exec[3] = {nullptr, nullptr, nullptr}; // start, iterations, update
  hipGraph_t graphs[3] = {nullptr, nullptr, nullptr};

  void drop_graphs()
  {
    for (int i = 0; i < 3; i++)
    {
      if (exec[i] != nullptr)
        (void)hipGraphExecDestroy(exec[i]);
      if (graphs[i] != nullptr)
        (void)hipGraphDestroy(graphs[i]);
      exec[i] = nullptr;
      graphs[i] = nullptr;
    }
  }

  ~akm_batch_s()
  {
    drop_graphs();
    if (stream != nullptr)
      (void)hipStreamDestroy(stream);
    if (host_state != nullptr)
      (void)hipHostFree(host_state);
  }

  int apply_all(int phase, int joff)
  {
    for (auto &w : walks)
      AKM_TRY(launch_fibre_batch(w.tpb, w.groups, fsys.data(), w.items.data(), jcol.data(), joff,
                                 restart, active.data(), phase, stream));
    for (auto &gr : groups)
      AKM_TRY(launch_rows_batch(gr.d, gr.n, gr.waves, args.data(), vsys.data(), gr.work.data(),
                                gr.nwork, gr.grid, jcol.data(), joff, restart, active.data(),
                                phase, stream));
    return AKM_SUCCESS;
  }

  int enqueue_start()
  {
    bt_begin<<<(nsys + 255) / 256, 256, 0, stream>>>(nsys, state.data(), active.data(),
                                                     open_dev.data(), jcol.data());
    bt_copy_rhs<<<dot_blocks, bt_threads, 0, stream>>>(dot_sys.data(), sys.data(),
                                                       active.data());
    AKM_TRY(check_launch("batch start"));
    AKM_TRY(apply_all(0, 0));
    bt_sumsq<<<dot_blocks, bt_threads, 0, stream>>>(dot_sys.data(), sys.data(), active.data());
    bt_finish<<<nsys, bt_threads, 0, stream>>>(sys.data(), state.data(), active.data(),
                                               open_dev.data(), jcol.data(), 0, restart);
    return check_launch("batch residual");
  }

  int enqueue_iterations()
  {
    for (int i = 0; i < bt_chunk; i++)
    {
      AKM_TRY(apply_all(1, i));
      const dim3 dgrid(dot_blocks + nsys, (restart + bt_cols - 1) / bt_cols);
      bt_dots<<<dgrid, bt_threads, 0, stream>>>(dot_sys.data(), dot_blocks, sys.data(),
                                               state.data(), active.data(), open_dev.data(),
                                               jcol.data(), i, restart);
      bt_update<<<upd_blocks, bt_upd_threads, 0, stream>>>(upd_sys.data(), sys.data(),
                                                           active.data(), open_dev.data(),
                                                           jcol.data(), i, restart);
    }
    bt_finish<<<nsys, bt_threads, 0, stream>>>(sys.data(), state.data(), active.data(),
                                               open_dev.data(), jcol.data(), bt_chunk, restart);
    bt_advance<<<1, 64, 0, stream>>>(jcol.data(), bt_chunk);
    return check_launch("batch iterations");
  }

  int enqueue_finish()
  {
    bt_backsolve<<<nsys, 64, 0, stream>>>(sys.data(), state.data());
    bt_xupdate<<<upd_blocks, bt_upd_threads, 0, stream>>>(upd_sys.data(), sys.data(),
                                                          state.data());
    return check_launch("batch update");
  }

  int capture(int which)
  {
    AKM_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    int rc = (which == 0) ? enqueue_start()
                          : (which == 1) ? enqueue_iterations() : enqueue_finish();
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(stream, &graph);
    if (rc != AKM_SUCCESS)
    {
      if (graph != nullptr)
        (void)hipGraphDestroy(graph);
      return rc;
    }
    if (e != hipSuccess)
      return set_error(AKM_ERR_HIP, "batch: graph capture failed: %s", hipGetErrorString(e));
    graphs[which] = graph;
    AKM_HIP(hipGraphInstantiate(&exec[which], graph, nullptr, nullptr, 0));
    return AKM_SUCCESS;
  }

  int plan_applies();

  //! The states on the host; open = systems still iterating.
  int read_state(int &open)
  {
    AKM_HIP(hipMemcpyAsync(host_state, state.data(), sizeof(bt_state) * nsys,
                           hipMemcpyDeviceToHost, stream));
    AKM_HIP(hipStreamSynchronize(stream));
    open = 0;
    for (int q = 0; q < nsys; q++)
      open += host_state[q].open;
    return AKM_SUCCESS;
  }

  //! The caller's vectors in (and the |b|^2 partials), or the solutions out.
  int move_vectors(double *const *x, const double *const *rhs, bool in)
  {
    for (int s0 = 0; s0 < nsys; s0 += bt_vectors)
    {
      const int s1 = std::min(nsys, s0 + bt_vectors);
      bt_io io{};
      io.first = s0;
      for (int q = s0; q < s1; q++)
      {
        io.x[q - s0] = x[q];
        io.b[q - s0] = rhs[q];
      }
      const int blocks = dot0[s1] - dot0[s0];
      if (in)
        bt_load<<<blocks, bt_threads, 0, stream>>>(dot_sys.data(), dot0[s0], sys.data(), io);
      else
        bt_store<<<blocks, bt_threads, 0, stream>>>(dot_sys.data(), dot0[s0], sys.data(), io);
    }
    return check_launch("batch vectors");
  }
};

static int time_group(akm_batch_s &b, akm_batch_s::group &gr, int waves, double &ms)
{
  hipEvent_t e0, e1;
  AKM_HIP(hipEventCreate(&e0));
  AKM_HIP(hipEventCreate(&e1));
  auto run = [&]() {
    return launch_rows_batch(gr.d, gr.n, waves, b.args.data(), b.vsys.data(), gr.work.data(),
                             gr.nwork, gr.grid, b.jcol.data(), 0, b.restart, b.active.data(), 0,
                             b.stream);
  };
  int rc = run();
  if (rc == AKM_SUCCESS)
  {
    (void)hipEventRecord(e0, b.stream);
    for (int r = 0; r < 3 && rc == AKM_SUCCESS; r++)
      rc = run();
    (void)hipEventRecord(e1, b.stream);
    (void)hipEventSynchronize(e1);
    float f = 0;
    (void)hipEventElapsedTime(&f, e0, e1);
    ms = f / 3.0;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

//! Chooses how every system is applied (for the forms its matrix has now),
//! tunes the pair groups on their work lists (X and V are overwritten) and
//! captures the graphs.
int akm_batch_s::plan_applies()
{
  drop_graphs();
  groups.clear();
  walks.clear();
  plans.clear();
  plans.resize(nsys);
  forms.clear();
  std::map<std::pair<int, int>, std::vector<int>> by_dn;
  std::map<int, std::vector<std::pair<int64_t, int2>>> by_tpb; // (length, item)
  std::vector<fibre_system> hf(nsys);
  for (int s = 0; s < nsys; s++)
  {
    akm_matrix m = mats[s];
    forms.push_back(m->form_stamp);
    int rc = AKM_SUCCESS;
    if (factored_batch_plan(*m, plans[s], rc))
    {
      hf[s] = fibre_batch_system(*m, plans[s], host_vsys[s].V, host_vsys[s].X, host_vsys[s].n,
                                 host_vsys[s].dt);
      // groups of slots come longest first within a system
      auto &items = by_tpb[plans[s].tpb];
      const int ng = plans[s].stages[0].groups;
      for (int g = 0; g < ng; g++)
        items.push_back({ng - g, make_int2(s, plans[s].stages[0].first_group + g)});
      continue;
    }
    AKM_TRY(rc);
    by_dn[{m->d, m->n}].push_back(s);
  }
  AKM_TRY(fsys.upload(hf.data(), nsys));
  // the largest workgroups, which run longest, first
  for (auto it = by_tpb.rbegin(); it != by_tpb.rend(); ++it)
  {
    auto &items = it->second;
    std::stable_sort(items.begin(), items.end(),
                     [](auto const &x, auto const &y) { return x.first > y.first; });
    std::vector<int2> list(items.size());
    for (size_t i = 0; i < items.size(); i++)
      list[i] = items[i].second;
    walk w;
    w.tpb = it->first;
    w.groups = static_cast<int>(list.size());
    AKM_TRY(w.items.upload(list.data(), int64_t(list.size())));
    walks.push_back(std::move(w));
  }
  // (d, n) groups with a longest-row-first work list over all their systems
  for (auto &kv : by_dn)
  {
    group gr;
    gr.d = kv.first.first;
    gr.n = kv.first.second;
    std::vector<std::pair<int64_t, int2>> items;
    for (int s : kv.second)
    {
      const auto &pn = mats[s]->pntr;
      for (int r = 0; r < mats[s]->rows; r++)
        items.push_back({pn[r + 1] - pn[r], make_int2(s, r)});
    }
    std::stable_sort(items.begin(), items.end(),
                     [](auto const &x, auto const &y) { return x.first > y.first; });
    std::vector<int2> w(items.size());
    for (size_t i = 0; i < items.size(); i++)
      w[i] = items[i].second;
    gr.nwork = static_cast<int>(w.size());
    gr.grid = std::min(gr.nwork, 4096);
    AKM_TRY(gr.work.upload(w.data(), int64_t(w.size())));
    groups.push_back(std::move(gr));
  }
  // autotune the workgroup shape of every pair group on its own work list
  if (!groups.empty())
  {
    const int zero = 0;
    const std::vector<int> ones(nsys, 1);
    AKM_TRY(jcol.upload(&zero, 1));
    AKM_TRY(active.upload(ones.data(), nsys));
    bt_fill<<<256, bt_threads, 0, stream>>>(total_n, X.data(), 0.5);
    bt_fill<<<256, bt_threads, 0, stream>>>(V.size(), V.data(), 0.0);
    AKM_TRY(check_launch("batch init"));
    for (auto &gr : groups)
    {
      double best = 1e300;
      int bw = 4;
      for (int w : {1, 2, 4, 8})
      {
        double ms = 0;
        AKM_TRY(time_group(*this, gr, w, ms));
        if (ms < best)
        {
          best = ms;
          bw = w;
        }
      }
      gr.waves = bw;
    }
    AKM_HIP(hipStreamSynchronize(stream));
  }
  std::map<std::pair<int, int>, int> waves;
  for (akm_matrix m : mats)
    waves[{m->d, m->n}] = 1;
  for (auto const &gr : groups)
    waves[{gr.d, gr.n}] = gr.waves;
  waves_of_dn.clear();
  for (auto const &kv : waves)
    waves_of_dn.push_back(kv.second);
  for (int i = 0; i < 3; i++)
    AKM_TRY(capture(i));
  return AKM_SUCCESS;
}

extern "C" {

akm_status akm_batch_create(int count, const akm_matrix *mats, const double *dts, int restart,
                            akm_batch *out)
{
  if (out == nullptr || mats == nullptr || dts == nullptr || count < 1)
    return set_error(AKM_ERR_INVALID, "batch: invalid arguments");
  *out = nullptr;
  auto b = std::make_unique<akm_batch_s>();
  b->nsys = count;
  AKM_HIP(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
  for (int s = 0; s < count; s++)
  {
    akm_matrix m = mats[s];
    if (m == nullptr || m->prec != AKM_F64 || m->mode != mode_grid || m->rows != m->cols ||
        m->rows < 1)
      return set_error(AKM_ERR_INVALID,
                       "batch: system %d must be a non-empty square FP64 sparse-grid matrix", s);
    if (!(m->n >= 2 && m->n <= 4 && m->d >= 1 && m->d <= 6) || (m->d == 6 && m->n > 2) ||
        (m->d >= 4 && m->n > 3))
      return set_error(AKM_ERR_UNSUPPORTED, "batch: (d, n) = (%d, %d) of system %d", m->d, m->n,
                       s);
  }
  int64_t min_n = mats[0]->output_size();
  for (int s = 0; s < count; s++)
    min_n = std::min<int64_t>(min_n, mats[s]->output_size());
  if (restart <= 0)
    restart = 50;
  restart = static_cast<int>(
      std::min<int64_t>({int64_t(restart), min_n, int64_t(bt_max_restart)}));
  b->restart = restart;
  b->mats.assign(mats, mats + count);

  // vector and block layout: dot-product blocks of 512 rows or a 256th of the
  // system, update blocks of one tile or a 512th
  std::vector<bt_sys> hs(count);
  std::vector<int> dot_sys, upd_sys;
  const int64_t m1 = restart;
  const int64_t small_per = 5 * (m1 + 2) + m1 * (m1 + 1) / 2 + 2;
  int64_t vtot = 0, small_tot = 0;
  for (int s = 0; s < count; s++)
  {
    bt_sys &q = hs[s];
    const int64_t n = mats[s]->output_size();
    b->n_of.push_back(n);
    b->x_off.push_back(b->total_n);
    q.n = n;
    q.drows = std::max<int64_t>(512, (n + 255) / 256);
    q.urows = std::max<int64_t>(1, (n + 512 * bt_tile - 1) / (512 * bt_tile)) * bt_tile;
    q.ndot = static_cast<int>((n + q.drows - 1) / q.drows);
    q.nupd = static_cast<int>((n + q.urows - 1) / q.urows);
    q.dot0 = static_cast<int>(dot_sys.size());
    q.upd0 = static_cast<int>(upd_sys.size());
    dot_sys.insert(dot_sys.end(), q.ndot, s);
    upd_sys.insert(upd_sys.end(), q.nupd, s);
    b->total_n += n;
    vtot += n * (restart + 1);
    small_tot += small_per + (m1 + 1) * q.ndot + std::max(q.ndot, q.nupd);
  }
  b->dot_blocks = static_cast<int>(dot_sys.size());
  b->upd_blocks = static_cast<int>(upd_sys.size());
  AKM_TRY(b->V.allocate(vtot));
  AKM_TRY(b->X.allocate(b->total_n));
  AKM_TRY(b->B.allocate(b->total_n));
  AKM_TRY(b->small.allocate(small_tot));
  {
    int64_t vo = 0, so = 0;
    for (int s = 0; s < count; s++)
    {
      bt_sys &q = hs[s];
      q.V = b->V.data() + vo;
      q.X = b->X.data() + b->x_off[s];
      q.B = b->B.data() + b->x_off[s];
      q.h = b->small.data() + so;
      q.H = q.h + (m1 + 1);
      q.cs = q.H + m1 * (m1 + 1) / 2 + 1;
      q.sn = q.cs + (m1 + 1);
      q.g = q.sn + (m1 + 1);
      q.inv = q.g + (m1 + 2);
      q.dotp = q.inv + (m1 + 2);
      q.sqp = q.dotp + (m1 + 1) * q.ndot;
      vo += q.n * (m1 + 1);
      so += small_per + (m1 + 1) * q.ndot + std::max(q.ndot, q.nupd);
    }
  }
  AKM_TRY(b->sys.upload(hs.data(), count));
  AKM_TRY(b->dot_sys.upload(dot_sys.data(), int64_t(dot_sys.size())));
  AKM_TRY(b->upd_sys.upload(upd_sys.data(), int64_t(upd_sys.size())));
  std::vector<kron_args<double>> ha(count);
  std::vector<batch_system> hv(count);
  for (int s = 0; s < count; s++)
  {
    ha[s] = kron_args_f64(*mats[s]);
    hv[s] = batch_system{hs[s].V, hs[s].X, hs[s].n, dts[s]};
  }
  AKM_TRY(b->args.upload(ha.data(), count));
  AKM_TRY(b->vsys.upload(hv.data(), count));
  b->host_vsys = std::move(hv);
  std::vector<bt_state> st0(count, bt_state{});
  AKM_TRY(b->state.upload(st0.data(), count));
  std::vector<int> ones(count, 1);
  AKM_TRY(b->active.upload(ones.data(), count));
  AKM_TRY(b->open_dev.upload(ones.data(), count));
  int zero = 0;
  AKM_TRY(b->jcol.upload(&zero, 1));
  AKM_HIP(hipHostMalloc(reinterpret_cast<void **>(&b->host_state), sizeof(bt_state) * count,
                        hipHostMallocDefault));
  for (bt_sys const &q : hs)
    b->dot0.push_back(q.dot0);
  b->dot0.push_back(b->dot_blocks);
  AKM_TRY(b->plan_applies());
  *out = b.release();
  return AKM_SUCCESS;
}

akm_status akm_batch_info(akm_batch b, int *restart, int *num_groups, int *group_waves)
{
  if (b == nullptr)
    return set_error(AKM_ERR_INVALID, "batch: null handle");
  if (restart)
    *restart = b->restart;
  if (num_groups)
    *num_groups = static_cast<int>(b->waves_of_dn.size());
  if (group_waves)
    std::copy(b->waves_of_dn.begin(), b->waves_of_dn.end(), group_waves);
  return AKM_SUCCESS;
}

akm_status akm_batch_solve(akm_batch b, double *const *x, const double *const *rhs,
                           int max_cycles, double tol, double *rel_residual, int *iterations,
                           int *converged)
{
  if (b == nullptr || x == nullptr || rhs == nullptr)
    return set_error(AKM_ERR_INVALID, "batch: null argument");
  if (tol <= 0)
    tol = 1e-10;
  if (max_cycles <= 0)
    max_cycles = 1000;
  hipStream_t s = b->stream;
  // x and b may come from any stream of the caller
  AKM_HIP(hipDeviceSynchronize());
  // new factors since the last solve: other products, or other values
  bool same = true;
  for (int q = 0; q < b->nsys; q++)
    same = same && b->forms[q] == b->mats[q]->form_stamp;
  if (!same)
    AKM_TRY(b->plan_applies());
  for (int q = 0; q < b->nsys; q++)
    if (b->plans[q].built)
      AKM_TRY(fibre_refresh(*b->mats[q], b->plans[q], s));
  for (int q = 0; q < b->nsys; q++)
    if (x[q] == nullptr || rhs[q] == nullptr)
      return set_error(AKM_ERR_INVALID, "batch: null vector of system %d", q);
  AKM_TRY(b->move_vectors(x, rhs, true));
  // tolerances from |b|
  bt_set_tol<<<b->nsys, 64, 0, s>>>(b->sys.data(), b->state.data(), tol);
  AKM_TRY(check_launch("batch tolerance"));
  int cycles = 0;
  bool all_done = false;
  while (true)
  {
    AKM_HIP(hipGraphLaunch(b->exec[0], s));
    int open = 0;
    AKM_TRY(b->read_state(open));
    if (open == 0)
    {
      all_done = true;
      break;
    }
    if (cycles >= max_cycles)
      break;
    // Arnoldi iterations, bt_chunk per replay, between host reads of the
    // per-system flags: a system that converges inside a chunk has cleared
    // its own flag, and the kernels skip it from then on
    for (int j = 0; j < b->restart; j += bt_chunk)
    {
      AKM_HIP(hipGraphLaunch(b->exec[1], s));
      AKM_TRY(b->read_state(open));
      if (open == 0)
        break;
    }
    AKM_HIP(hipGraphLaunch(b->exec[2], s));
    ++cycles;
  }
  AKM_TRY(b->move_vectors(x, rhs, false));
  AKM_HIP(hipStreamSynchronize(s)); // the solutions are in x; host_state is the last read
  for (int q = 0; q < b->nsys; q++)
  {
    const bt_state &t = b->host_state[q];
    const double bn = (tol > 0) ? t.tol / tol : 0.0;
    if (rel_residual)
      rel_residual[q] = (bn > 0) ? t.res / bn : t.res;
    if (iterations)
      iterations[q] = t.iters;
    if (converged)
      converged[q] = t.converged;
  }
  return all_done ? AKM_SUCCESS : AKM_ERR_NOT_CONVERGED;
}

akm_status akm_batch_destroy(akm_batch b)
{
  if (b != nullptr)
    (void)hipStreamSynchronize(b->stream);
  delete b;
  return AKM_SUCCESS;
}

} // extern "C"
