// Global Kronecker operator: the reference's default single-node kronmult
// mode (global_kron_matrix, src/asgard_kronmult_matrix.hpp:780-989,
// src/asgard_kronmult_matrix.cpp:1008-1590), on the GPU.
//
// The operator sum_t (A_t0 x ... x A_t,d-1) restricted to the grid's DOFs is
// applied one dimension at a time.  Every term with k non-identity factors
// becomes 2^(k-1) chains of k one-dimensional products over the cell set
// completed with its missing ancestors ("padded"); in each chain the upper
// parts (diagonal included) of some factors act first, one factor acts whole,
// and the strictly lower parts of the others act last
// (src/device/asgard_kronmult.hpp:152-220).  On a set closed under taking
// ancestors in every dimension this reproduces the pair-by-pair operator
// exactly for hierarchical (volume) couplings, and for every coupling on
// standard sparse grids.
//
// GPU layout: DOF vectors keep the pair operator's layout (cell-major, n^d
// tensor per cell, dimension 0 slowest), padded cells appended after the
// active ones.  For every dimension k and cell the host lists the connected
// cells of its fibre (cells equal in all other 1D indices) with their
// connect_1d positions.  A one-dimensional product in dimension k runs in
// one of these layouts, which akm_autotune times: one lane per (chain, DOF),
// the lanes of a cell reading each connected cell's tensor together; one
// wavefront per (chain, cell) whose lane groups split the list; the fibre
// walk (layout 8, fibre.hip), whose slots split every list into short pieces
// and which takes the products shared by chains once; or the slab layout
// below.
// Cells are taken fibre by fibre, so the cells reading the same tensors run
// together.  The factor values are the same connect_1d blocks (vA) the pair
// operator uses.  All chains advance together, one launch per stage, each
// chain in its own ping-pong slot; one more launch sums the chains in chain
// order and applies alpha/beta/gamma (and optionally the reference's Jacobi
// scaling).
#include "akm_internal.hpp"
#include "fibre.hpp"
#include "grid.hpp"
#include "matrix.hpp"

#include <algorithm>
#include <map>
#include <memory>
#include <vector>

namespace akm
{
constexpr int gk_max_dims = 6;
constexpr int gk_threads = 256;
constexpr int gk_group_max = 4; // chains sharing one first-stage input read

//! Device view of the global operator.
struct gk_args
{
  int d, n, N, T;
  int64_t active_cells, cells; // active first, then padding
  const int *elem;             // cells x d 1D indices
  // per dimension: every cell's connected cells of its fibre (cells equal in
  // all other 1D indices), 1D index ascending, with their connect_1d position
  const int *nb_ptr[gk_max_dims];  // cells + 1
  const int *nb_cell[gk_max_dims];
  const int *nb_q[gk_max_dims];
  const int *nb_diag[gk_max_dims]; // position of the cell itself
  const int *order[gk_max_dims];   // cells fibre by fibre (processing order)
  const int *ch_term;  // chain -> term
  const int *ch_nst;   // chain -> number of stages
  const int *ch_dim;   // chain -> dims of its stages (gk_max_dims each)
  const int *ch_fill;  // chain -> fills of its stages
  const int *ch_slot;  // chain -> work-buffer slot (-1 for identity-only terms)
  int nchains;
  int nslots;          // chains with at least one stage
  int64_t stride;      // work-buffer slot size (padded DOFs)
  bool xcd_order;      // cell layouts: each XCD takes contiguous items
};

//! One stage's product for DOF i of a chain: (fill part of A_{t,k}) applied
//! along dimension k to `in` (padded vector, or the active-only x when
//! `in_active_only`).  The lanes of a cell read each connected cell's tensor
//! together (coalesced).
template<typename P>
__device__ __forceinline__ P gk_row_part(gk_args const &a, const P *__restrict__ vA, int t,
                                         int k, int fill, const P *__restrict__ in,
                                         bool in_active_only, int64_t i)
{
  const int N = a.N, n = a.n, d = a.d;
  const int64_t cell = i / N;
  const int e = static_cast<int>(i - cell * N);
  int stride_k = 1;
  for (int j = k + 1; j < d; j++)
    stride_k *= n;
  const int s = (e / stride_k) % n;
  const int e0 = e - s * stride_k;
  const int dg = a.nb_diag[k][cell];
  const int lo = (fill == gk_upper) ? dg : a.nb_ptr[k][cell];
  const int hi = (fill == gk_lower) ? dg + 1 : a.nb_ptr[k][cell + 1];
  const int64_t nn = int64_t(n) * n;
  const int64_t tstride = int64_t(d) * nn;
  const int64_t cstride = tstride * a.T;
  const P *Ab = vA + int64_t(t) * tstride + k * nn + s;
  const int *__restrict__ ncell = a.nb_cell[k];
  const int *__restrict__ nq = a.nb_q[k];
  P acc = 0;
#pragma unroll 4
  for (int p = lo; p < hi; p++)
  {
    const int cj = ncell[p];
    if (in_active_only && cj >= a.active_cells)
      continue;
    int jlo = 0, jhi = n;
    if (p == dg)
    {
      if (fill == gk_upper)
        jlo = s;
      else if (fill == gk_lower)
        jhi = s;
    }
    const P *A = Ab + int64_t(nq[p]) * cstride; // A[j*n] = A(s, j)
    const P *xin = in + int64_t(cj) * N + e0;
    for (int j = jlo; j < jhi; j++)
      acc = fma(A[j * n], xin[j * stride_k], acc);
  }
  return acc;
}

//! Stage `st` of every chain with more than st stages; one lane per (chain,
//! padded DOF), cells taken fibre by fibre so that the cells reading the same
//! connected tensors run together.
template<typename P>
__global__ void __launch_bounds__(gk_threads)
    gk_stage(gk_args a, const P *__restrict__ vA, const int *__restrict__ list, int nlist, int st,
             const P *__restrict__ x, P *work)
{
  const int64_t dofs = a.cells * a.N;
  const int64_t count = dofs * nlist;
  for (int64_t gi = blockIdx.x * int64_t(gk_threads) + threadIdx.x; gi < count;
       gi += int64_t(gk_threads) * gridDim.x)
  {
    const int li = static_cast<int>(gi / dofs);
    const int64_t pos = gi - int64_t(li) * dofs;
    const int c = list[li];
    const int slot = a.ch_slot[c];
    const int k = a.ch_dim[c * gk_max_dims + st];
    const int64_t pcell = pos / a.N;
    const int64_t i = int64_t(a.order[k][pcell]) * a.N + (pos - pcell * a.N);
    const int fill = a.ch_fill[c * gk_max_dims + st];
    const P *in = (st == 0) ? x : work + (int64_t((st - 1) & 1) * a.nslots + slot) * a.stride;
    work[(int64_t(st & 1) * a.nslots + slot) * a.stride + i] =
        gk_row_part<P>(a, vA, a.ch_term[c], k, fill, in, st == 0, i);
  }
}

//! Cell layout: one wavefront per (chain, cell).  Lane (g, e), e < N, g <
//! 64/N, takes every (64/N)-th connection of the cell's list starting at g;
//! the lanes of one g read a connected cell's tensor together, and the list
//! itself is loaded 64 entries at a time and passed between lanes.  Two
//! connections are fetched before either is used (compile-time n = NT; NT = 0
//! reads n at run time; two keeps the kernel at 5+ wavefronts per SIMD, four
//! measured slower).  Returns this lane's partial sum for entry e (0 on
//! idle lanes).
template<typename P, int NT>
__device__ __forceinline__ P gk_cell_part(gk_args const &a, const P *__restrict__ vA, int t, int k,
                                          int fill, const P *__restrict__ in, bool in_active_only,
                                          int64_t cell, int lane)
{
  constexpr int U = 2;
  const int N = a.N, d = a.d;
  const int n = (NT > 0) ? NT : a.n;
  const int G = wave_size / N;
  const int g = lane / N;
  const int e = lane - g * N;
  int stride_k = 1;
  for (int j = k + 1; j < d; j++)
    stride_k *= n;
  const int s = (e / stride_k) % n;
  const int e0 = e - s * stride_k;
  const int dg = a.nb_diag[k][cell];
  const int lo = (fill == gk_upper) ? dg : a.nb_ptr[k][cell];
  const int hi = (fill == gk_lower) ? dg + 1 : a.nb_ptr[k][cell + 1];
  const int64_t nn = int64_t(n) * n;
  const int64_t tstride = int64_t(d) * nn;
  const int64_t cstride = tstride * a.T;
  const P *Ab = vA + int64_t(t) * tstride + k * nn + s;
  P acc = 0;
  for (int base = lo; base < hi; base += wave_size)
  {
    const int pl = base + lane;
    const int my_cj = (pl < hi) ? a.nb_cell[k][pl] : 0;
    const int my_q = (pl < hi) ? a.nb_q[k][pl] : 0;
    const int cnt = min(wave_size, hi - base);
    // the same trip count on every lane: the shuffles run with the whole
    // wavefront active (a shuffle from an inactive lane reads zero)
    const int iters = (cnt + G - 1) / G;
    for (int it = 0; it < iters; it += U)
    {
      int cjv[U], qv[U], jlov[U], jhiv[U];
#pragma unroll
      for (int u = 0; u < U; u++)
      {
        const int r = (it + u) * G + g;
        const int rr = min(r, wave_size - 1);
        const int cj = __shfl(my_cj, rr, wave_size);
        const int q = __shfl(my_q, rr, wave_size);
        const bool ok =
            (it + u < iters) && g < G && r < cnt && !(in_active_only && cj >= a.active_cells);
        const bool diag = ok && (base + r == dg);
        // idle entries read cell 0 / connection 0 (valid addresses) and add nothing
        cjv[u] = ok ? cj : 0;
        qv[u] = ok ? q : 0;
        jlov[u] = (diag && fill == gk_upper) ? s : 0;
        jhiv[u] = !ok ? 0 : ((diag && fill == gk_lower) ? s : n);
      }
      if constexpr (NT > 0)
      {
        P av[U][NT], xv[U][NT];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int j = 0; j < NT; j++)
          {
            av[u][j] = Ab[int64_t(qv[u]) * cstride + j * NT];
            xv[u][j] = in[int64_t(cjv[u]) * N + e0 + j * stride_k];
          }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int j = 0; j < NT; j++)
          {
            const P v = fma(av[u][j], xv[u][j], acc);
            acc = (j >= jlov[u] && j < jhiv[u]) ? v : acc;
          }
      }
      else
      {
        for (int u = 0; u < U; u++)
        {
          const P *A = Ab + int64_t(qv[u]) * cstride;
          const P *xin = in + int64_t(cjv[u]) * N + e0;
          for (int j = jlov[u]; j < jhiv[u]; j++)
            acc = fma(A[j * n], xin[j * stride_k], acc);
        }
      }
    }
  }
  return acc;
}

//! Orders the LDS accesses of one wavefront (no workgroup barrier needed).
__device__ __forceinline__ void gk_wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

//! Sums the wavefront's partials over g in order into lanes g = 0 (LDS
//! slice of wave_size values owned by this wavefront).
template<typename P>
__device__ __forceinline__ P gk_cell_reduce(P v, P *red, int lane, int N)
{
  if (N == wave_size)
    return v; // one lane group: nothing to add
  red[lane] = v;
  gk_wave_sync();
  P sum = 0;
  if (lane < N)
    for (int g = 0; g < wave_size / N; g++)
      sum += red[g * N + lane];
  gk_wave_sync();
  return sum;
}

//! Workgroup index with the workgroups of one XCD made consecutive: the
//! hardware deals workgroups round-robin over the 8 XCDs, so workgroups
//! b, b + 8, b + 16, ... share an L2.  With the grid a multiple of 8 this is
//! a permutation, and the waves of one XCD take contiguous items (cells of
//! the same fibres), whose neighbours then hit that XCD's L2.
__device__ __forceinline__ int64_t gk_xcd_block(bool on)
{
  constexpr int xcds = 8;
  const int per = gridDim.x / xcds;
  return (on && per * xcds == static_cast<int>(gridDim.x))
             ? int64_t(blockIdx.x % xcds) * per + blockIdx.x / xcds
             : int64_t(blockIdx.x);
}

//! Stage `st` in the cell layout.
template<typename P, int NT>
__global__ void __launch_bounds__(gk_threads)
    gk_cell_stage(gk_args a, const P *__restrict__ vA, const int *__restrict__ list, int nlist,
                  int st, const P *__restrict__ x, P *work)
{
  __shared__ P red[gk_threads];
  const int lane = threadIdx.x % wave_size;
  P *wred = red + (threadIdx.x / wave_size) * wave_size;
  const int64_t items = a.cells * nlist;
  for (int64_t w = (gk_xcd_block(a.xcd_order) * gk_threads + threadIdx.x) / wave_size; w < items;
       w += int64_t(gk_threads / wave_size) * gridDim.x)
  {
    const int li = static_cast<int>(w / a.cells);
    const int c = list[li];
    const int slot = a.ch_slot[c];
    const int k = a.ch_dim[c * gk_max_dims + st];
    const int64_t cell = a.order[k][w - int64_t(li) * a.cells];
    const P *in = (st == 0) ? x : work + (int64_t((st - 1) & 1) * a.nslots + slot) * a.stride;
    const P v = gk_cell_reduce(gk_cell_part<P, NT>(a, vA, a.ch_term[c], k,
                                               a.ch_fill[c * gk_max_dims + st], in, st == 0,
                                               cell, lane),
                               wred, lane, a.N);
    if (lane < a.N)
      work[(int64_t(st & 1) * a.nslots + slot) * a.stride + cell * a.N + lane] = v;
  }
}

//! gk_cell_part for a group of chains whose stage reads the same input
//! along the same dimension with the same fill (the first stage of chains of
//! different terms): the input values are loaded once per connection and
//! each chain's factor block is applied to them.  Every chain's sum is
//! formed in the same order as gk_cell_part forms it.
template<typename P, int NT, int GM>
__device__ __forceinline__ void gk_cell_part_group(gk_args const &a, const P *__restrict__ vA,
                                                   const int (&tg)[GM], int gm, int k, int fill,
                                                   const P *__restrict__ in, int64_t cell,
                                                   int lane, P (&acc)[GM])
{
  constexpr int U = 2;
  const int N = a.N, d = a.d;
  const int G = wave_size / N;
  const int g = lane / N;
  const int e = lane - g * N;
  int stride_k = 1;
  for (int j = k + 1; j < d; j++)
    stride_k *= NT;
  const int s = (e / stride_k) % NT;
  const int e0 = e - s * stride_k;
  const int dg = a.nb_diag[k][cell];
  const int lo = (fill == gk_upper) ? dg : a.nb_ptr[k][cell];
  const int hi = (fill == gk_lower) ? dg + 1 : a.nb_ptr[k][cell + 1];
  const int64_t nn = int64_t(NT) * NT;
  const int64_t tstride = int64_t(d) * nn;
  const int64_t cstride = tstride * a.T;
  const P *Ab[GM];
#pragma unroll
  for (int m = 0; m < GM; m++)
  {
    acc[m] = 0;
    // members past gm repeat the first chain's (valid) blocks; their sums are dropped
    Ab[m] = vA + int64_t(tg[m < gm ? m : 0]) * tstride + k * nn + s;
  }
  for (int base = lo; base < hi; base += wave_size)
  {
    const int pl = base + lane;
    const int my_cj = (pl < hi) ? a.nb_cell[k][pl] : 0;
    const int my_q = (pl < hi) ? a.nb_q[k][pl] : 0;
    const int cnt = min(wave_size, hi - base);
    const int iters = (cnt + G - 1) / G;
    for (int it = 0; it < iters; it += U)
    {
      int cjv[U], qv[U], jlov[U], jhiv[U];
#pragma unroll
      for (int u = 0; u < U; u++)
      {
        const int r = (it + u) * G + g;
        const int rr = min(r, wave_size - 1);
        const int cj = __shfl(my_cj, rr, wave_size);
        const int q = __shfl(my_q, rr, wave_size);
        const bool ok = (it + u < iters) && g < G && r < cnt && cj < a.active_cells;
        const bool diag = ok && (base + r == dg);
        cjv[u] = ok ? cj : 0;
        qv[u] = ok ? q : 0;
        jlov[u] = (diag && fill == gk_upper) ? s : 0;
        jhiv[u] = !ok ? 0 : ((diag && fill == gk_lower) ? s : NT);
      }
      P xv[U][NT];
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int j = 0; j < NT; j++)
          xv[u][j] = in[int64_t(cjv[u]) * N + e0 + j * stride_k];
#pragma unroll
      for (int m = 0; m < GM; m++)
      {
        if (m >= gm) // the same on every lane
          break;
        P av[U][NT];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int j = 0; j < NT; j++)
            av[u][j] = Ab[m][int64_t(qv[u]) * cstride + j * NT];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
          for (int j = 0; j < NT; j++)
          {
            const P v = fma(av[u][j], xv[u][j], acc[m]);
            acc[m] = (j >= jlov[u] && j < jhiv[u]) ? v : acc[m];
          }
      }
    }
  }
}

//! The first stage in the cell layout with chains grouped by (dimension,
//! fill): one wavefront per (group, cell) reads the neighbours' x values once
//! for up to GM chains.  Group gi holds chains gchain[gptr[gi] .. gptr[gi+1]).
template<typename P, int NT, int GM>
__global__ void __launch_bounds__(gk_threads)
    gk_cell_first(gk_args a, const P *__restrict__ vA, const int *__restrict__ gptr,
                  const int *__restrict__ gchain, int ngroups, const P *__restrict__ x, P *work)
{
  __shared__ P red[gk_threads];
  const int lane = threadIdx.x % wave_size;
  P *wred = red + (threadIdx.x / wave_size) * wave_size;
  const int64_t items = a.cells * ngroups;
  for (int64_t w = (gk_xcd_block(a.xcd_order) * gk_threads + threadIdx.x) / wave_size; w < items;
       w += int64_t(gk_threads / wave_size) * gridDim.x)
  {
    const int gi = static_cast<int>(w / a.cells);
    const int g0 = gptr[gi], gm = gptr[gi + 1] - g0;
    const int c0 = gchain[g0];
    const int k = a.ch_dim[c0 * gk_max_dims];
    const int fill = a.ch_fill[c0 * gk_max_dims];
    const int64_t cell = a.order[k][w - int64_t(gi) * a.cells];
    int tg[GM];
#pragma unroll
    for (int m = 0; m < GM; m++)
      tg[m] = (m < gm) ? a.ch_term[gchain[g0 + m]] : 0;
    P acc[GM];
    gk_cell_part_group<P, NT, GM>(a, vA, tg, gm, k, fill, x, cell, lane, acc);
#pragma unroll
    for (int m = 0; m < GM; m++)
    {
      if (m < gm)
      {
        const P v = gk_cell_reduce(acc[m], wred, lane, a.N);
        if (lane < a.N)
          work[int64_t(a.ch_slot[gchain[g0 + m]]) * a.stride + cell * a.N + lane] = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Slab layout.  The terms with the same one or two non-identity dimensions S
// form a group.  A slab of the group is a class of cells equal in every 1D
// index outside S; every stage of the group's chains maps a slab into
// itself (a stage along k in S reads only the cell's fibre along k), so one
// workgroup loads a slab's x once, runs all the group's chains on it in LDS
// and writes the group's sum once.  Small slabs are bundled into one
// workgroup; a slab too large for LDS is split over the other-index
// combinations (the tensor entries outside S, on which the group's factors
// act as the identity).  Per pass the 1D factor blocks of one (term,
// dimension), restricted to the 1D indices below the bundle's level bound,
// and the bundle's connection lists along that dimension are staged in LDS
// as well, so the connection loops touch only LDS.

// a bundle holds at most 256 blocks (one per thread), a large slab alone up
// to 1024
constexpr int gs_blocks_small = 256;
//! Blocks of a small bundle tried first: FP64 bundles of 512 blocks (512
//! threads) measured faster than 256 on the d=6 Vlasov operator, FP32 ones
//! slower.  A group whose 512-block bundles do not fit LDS is planned again
//! with 256.
__host__ __device__ constexpr int gs_blocks_small_first(int esize)
{
  return esize == 8 ? 512 : gs_blocks_small;
}
constexpr int gs_blocks_large = 1024;
constexpr int gs_lds_max = 160 * 1024;
constexpr int gs_pad = 2; // values of padding after each cell's blocks in LDS
static_assert(gs_pad % 2 == 0, "pair-major FP64 blocks need cells an even count of values apart");
constexpr int gs_split_level = 5; // slabs with level bound >= this run one chain per workgroup
constexpr int gs_lds_resident = 64 * 1024; // stage everything at once up to this size
constexpr int gs_unroll = 8;               // independent loads per thread while staging

//! Consecutive slabs of one group, their cells in bundle-local order.
struct gs_bundle
{
  int group;
  int cell0;    // first entry in gs_args::cells
  int ncell;
  int C;        // other-index combinations per chunk
  int Lp;       // level bound of the slab dimensions (compact factor table)
  int resident; // 1: every factor table and both lists staged once
  int list0;    // first int of the bundle's list images in gs_args::lists
  int llen[2];  // per slab dimension: image length (starts, diagonals, entries)
};

//! A group: its slab dimensions, factor tables and passes.
struct gs_group
{
  int nd;           // slab dimensions (1 or 2)
  int dim[2];       // ascending
  int str[2];       // their strides in the cell tensor
  int call;         // other-index combinations, n^(d - nd)
  int off0;         // first of its call entries in gs_args::offs
  int tab0, ntab;   // its (term, dimension) factor tables in gs_args::tabs
  int pass0, npass; // its passes in gs_args::passes
  int slot;         // work-buffer slot of the group's sum
};

//! One pass: a chain's stage.  mode 0: x -> sum (one-stage chain); 1: x ->
//! intermediate; 2: intermediate -> sum; 3: the same stage of two chains at
//! once (the last of one, the first of the next), intermediate -> sum and x
//! -> intermediate.
struct gs_pass
{
  int tab;  // factor table index within the group
  int j;    // slab dimension index (0 or 1)
  int fill, mode;
};

//! A split item's pass and its lanes.
struct gs_lane_pass
{
  gs_pass ps;
  int slot0, nslot; // in gs_args::slots
  int rec0;         // their records in gs_args::recs
};

//! One workgroup's work: a chunk of a bundle with its group's data, so that
//! one record read starts it.
struct gs_item
{
  int cell0, ncell; // the bundle's cells in gs_args::cells
  int C;            // other-index combinations per chunk
  int cb, tstride;  // the group's first compact factor table in gs_ctab, values per table
  int resident;     // 1: every factor table and both lists staged once
  int list0;        // first int of the bundle's list images
  int llen[2];      // per slab dimension: image length
  int nd;           // slab dimensions (1 or 2)
  int str[2];       // their strides in the cell tensor
  int off;          // first of the chunk's C entries in gs_args::offs
  int ntab;         // the group's factor tables
  int pass0, npass; // the group's passes in gs_args::passes
  int slot;         // work-buffer slot of the group's sum
  // a split item (one chain of a large slab): its chain of the bundle's nch
  // and the bundle's first partial in the partial buffer (-1: not split);
  // cell c's partial of chain k is partial part + c * nch + k (N values);
  // its passes
  int part, nch, chain;
  gs_lane_pass pass[2];
};

struct gs_args
{
  int d, n, N, T;
  int64_t active_cells;
  int64_t stride; // work-buffer slot size
  const gs_pass *passes;
  const int *cells; // bundle cells (padded cell indices)
  // per bundle and slab dimension, the LDS image of its lists: ncell + 1
  // starts and ncell diagonal positions (relative to the entries), then
  // the entries (the connected cell's element offset in the bundle's x |
  // its factor block's element offset in the compact table << 16)
  const int *lists;
  const int *offs; // tensor offsets of the other-index combinations
  const int *slots; // split items' lanes: record | entry << 16 (-1: none)
  const int *recs;
};

//! Values of one compact factor table of nq n x n blocks, filled up to
//! whole 16 bytes of either precision.
__host__ __device__ inline int gs_table_values(int nq, int nn) { return (nq * nn + 3) / 4 * 4; }

//! LDS bytes of one work item: x (and the intermediate when nd = 2), ntab
//! factor tables of nq blocks, then the int lists (nlist_ints).
__host__ __device__ inline int64_t gs_lds_bytes(int esize, int nd, int n, int ncell, int C, int nq,
                                                int ntab, int64_t nlist_ints, int npass)
{
  const int64_t ds = (nd == 1) ? n : int64_t(n) * n;
  const int64_t bd = int64_t(ncell) * (ds * C + gs_pad);
  const int64_t vals = bd * nd + int64_t(ntab) * gs_table_values(nq, n * n);
  return int64_t(16) * npass + (vals * esize + 15) / 16 * 16 + 4 * nlist_ints;
}

//! The same of a split item: x, the intermediate, one factor table.
__host__ __device__ inline int64_t gs_split_lds(int esize, int nd, int n, int ncell, int C, int nq)
{
  const int64_t ds = (nd == 1) ? n : int64_t(n) * n;
  const int64_t bd = int64_t(ncell) * (ds * C + gs_pad);
  return (bd * nd * esize + 15) / 16 * 16 + int64_t(gs_table_values(nq, n * n)) * esize;
}

//! dst[i] = src[i], i < count, by a workgroup of TPB threads with
//! gs_unroll loads per thread in flight.
template<int TPB, typename T>
__device__ __forceinline__ void gs_copy(T *dst, const T *__restrict__ src, int count)
{
  // whole batches without bounds tests, then the remainder
  const int full = count / (gs_unroll * TPB) * (gs_unroll * TPB);
  for (int base = threadIdx.x; base < full; base += gs_unroll * TPB)
  {
    T v[gs_unroll];
#pragma unroll
    for (int u = 0; u < gs_unroll; u++)
      v[u] = src[base + u * TPB];
#pragma unroll
    for (int u = 0; u < gs_unroll; u++)
      dst[base + u * TPB] = v[u];
  }
  for (int base = full + threadIdx.x; base < count; base += gs_unroll * TPB)
  {
    T v[gs_unroll];
#pragma unroll
    for (int u = 0; u < gs_unroll; u++)
    {
      const int i = base + u * TPB;
      v[u] = (i < count) ? src[i] : T{};
    }
#pragma unroll
    for (int u = 0; u < gs_unroll; u++)
    {
      const int i = base + u * TPB;
      if (i < count)
        dst[i] = v[u];
    }
  }
}

//! One connection's block product along slab dimension J of ND: v[s] +=
//! sum_r A(s_J, r) * xb[s with s_J = r] over r in [rlo(s_J), rhi(s_J)): all
//! columns (FILL_FULL), from the row's own index on (upper diagonal block),
//! or before it (lower diagonal block).  Blocks are n^ND values, the last
//! slab digit fastest; A(s, r) = A[s + r * NT].
enum gs_cols : int
{
  gs_all = 0,
  gs_from_diag = 1,
  gs_before_diag = 2,
};

template<typename P, int NT, int ND, int J, int COLS>
__device__ __forceinline__ void gs_block_fma(const P (&av)[NT * NT],
                                             const P (&xv)[(ND == 1) ? NT : NT * NT], P *v)
{
  constexpr int ds = (ND == 1) ? NT : NT * NT;
#pragma unroll
  for (int si = 0; si < ds; si++)
  {
    const int s0 = (ND == 1) ? si : si / NT;
    const int s1 = (ND == 1) ? 0 : si % NT;
    const int sj = (J == 0) ? s0 : s1;
#pragma unroll
    for (int r = 0; r < NT; r++)
    {
      if ((COLS == gs_from_diag && r < sj) || (COLS == gs_before_diag && r >= sj))
        continue;
      const int xi = (ND == 1) ? r : ((J == 0) ? r * NT + s1 : s0 * NT + r);
      v[si] = fma(av[sj + r * NT], xv[xi], v[si]);
    }
  }
}

//! How a cell's blocks of DS values sit in LDS.  FP64 blocks with an even
//! value count are pair-major: values 2q and 2q + 1 of chunk entry o at
//! 2 (q C + o), one 16-byte read.  Other FP64 blocks are value-major (value
//! s of entry o at s C + o).  FP32 blocks are entry-major (DS o + s).  In
//! the FP64 orders a wavefront's lanes, which hold consecutive entries o,
//! read consecutive words instead of 32-byte strides, which spreads them
//! over the LDS banks; an FP32 block of four values is one 16-byte read.
template<typename P>
constexpr bool gs_value_major = sizeof(P) == 8;
template<typename P, int DS>
constexpr bool gs_pair_major = sizeof(P) == 8 && DS % 2 == 0;

//! The LDS offset of value si of a block whose entry starts at ob, with
//! value (pair, for pair-major blocks) stride vs.
template<typename P, int DS>
__device__ __forceinline__ int gs_at(int si, int ob, int vs)
{
  if constexpr (gs_pair_major<P, DS>)
    return ob + (si >> 1) * vs + (si & 1);
  else
    return ob + si * vs;
}

//! Where value w of block q sits in a compact factor table of nq blocks:
//! FP64 blocks of an even value count in planes of pairs, others in one
//! piece.
template<typename P>
__host__ __device__ inline int gs_table_at(int q, int w, int nq, int nn)
{
  return (sizeof(P) == 8 && nn % 2 == 0) ? (w / 2 * nq + q) * 2 + w % 2 : q * nn + w;
}

//! A block of DS values at xb, its values (pairs, when pair-major) vs apart.
template<typename P, int DS>
__device__ __forceinline__ void gs_x_load(const P *xb, int vs, P (&xv)[DS])
{
  if constexpr (gs_pair_major<P, DS>)
  {
#pragma unroll
    for (int q = 0; q < DS / 2; q++)
    {
      const double2 t = *reinterpret_cast<const double2 *>(xb + q * vs);
      xv[2 * q] = t.x;
      xv[2 * q + 1] = t.y;
    }
  }
  else
  {
#pragma unroll
    for (int k = 0; k < DS; k++)
      xv[k] = xb[k * vs];
  }
}

//! The factor block and the x block of one list entry: the block starts at
//! in + ob + the entry's cell offset, its values (pairs, when pair-major)
//! vs apart.  FP64 factor blocks of an even value count are read in 16-byte
//! pairs, each pair of the block in a plane of its own (gs_table_at), planes
//! `plane` values apart: lanes on neighbouring blocks then read neighbouring
//! words, where blocks in one piece (32 bytes for n = 2) left half the LDS
//! banks unused by each read (the operator above: 111 -> 103 us).
template<typename P, int NT, int ND>
__device__ __forceinline__ void gs_block_load(const P *tab, int plane, const P *in, unsigned e,
                                              int ob, int vs, P (&av)[NT * NT],
                                              P (&xv)[(ND == 1) ? NT : NT * NT])
{
  constexpr int ds = (ND == 1) ? NT : NT * NT;
  const P *A = tab + (e >> 16);
  const P *xb = in + (e & 0xffffu) + ob;
  if constexpr (gs_pair_major<P, NT * NT>)
  {
#pragma unroll
    for (int q = 0; q < NT * NT / 2; q++)
    {
      const double2 t = *reinterpret_cast<const double2 *>(A + q * plane);
      av[2 * q] = t.x;
      av[2 * q + 1] = t.y;
    }
  }
  else
  {
#pragma unroll
    for (int k = 0; k < NT * NT; k++)
      av[k] = A[k];
  }
  gs_x_load<P, ds>(xb, vs, xv);
}

//! One pass along slab dimension J for one block (cell c >= 0, block base
//! ob within the cell, values or pairs vs apart): the fill part of the
//! staged factor applied to `in`.
//! List entries hold the connected cell's element offset in `in` (low 16
//! bits) and its factor block's offset in `tab` (high 16 bits).  Each
//! value's sum runs over the connections ascending, then the factor's
//! columns, as in gk_cell_part; the diagonal block, restricted by the fill,
//! is the first connection of an upper fill and the last of a lower one.
//! The loop is software-pipelined: the blocks of the next connection and
//! the list entry after it are read while this connection's products run.
//! Two inputs of one pass (M = 2, in1 beside in) share the list entries and
//! factor blocks.
template<typename P, int NT, int ND, int J, int M>
__device__ __forceinline__ void gs_pass_block(const P *in, const P *in1, const P *tab, int plane,
                                              const int *st, const int *dg, const unsigned *ent,
                                              int c, int ob, int vs, int fill, P *v, P *v1)
{
  constexpr int ds = (ND == 1) ? NT : NT * NT;
  const int d0 = dg[c];
  const int lo = (fill == gk_upper) ? d0 + 1 : st[c];
  const int hi = (fill == gk_lower) ? d0 : st[c + 1];
  P av[NT * NT], xv[M][ds];
  auto load = [&](unsigned e, P(&a)[NT * NT], P(&b)[M][ds]) {
    gs_block_load<P, NT, ND>(tab, plane, in, e, ob, vs, a, b[0]);
    if constexpr (M == 2)
      gs_x_load<P, ds>(in1 + (e & 0xffffu) + ob, vs, b[1]);
  };
  auto apply = [&](auto cols) {
    gs_block_fma<P, NT, ND, J, cols.value>(av, xv[0], v);
    if constexpr (M == 2)
      gs_block_fma<P, NT, ND, J, cols.value>(av, xv[1], v1);
  };
  if (fill == gk_upper)
  {
    load(ent[d0], av, xv);
    apply(std::integral_constant<int, gs_from_diag>{});
  }
  if (lo < hi)
  {
    load(ent[lo], av, xv);
    unsigned en = ent[(lo + 1 < hi) ? lo + 1 : d0];
    for (int p = lo; p < hi; p++)
    {
      P an[NT * NT], xn[M][ds];
      load(en, an, xn);
      en = ent[(p + 2 < hi) ? p + 2 : d0];
      apply(std::integral_constant<int, gs_all>{});
#pragma unroll
      for (int k = 0; k < NT * NT; k++)
        av[k] = an[k];
#pragma unroll
      for (int m = 0; m < M; m++)
#pragma unroll
        for (int k = 0; k < ds; k++)
          xv[m][k] = xn[m][k];
    }
  }
  if (fill == gk_lower)
  {
    load(ent[d0], av, xv);
    apply(std::integral_constant<int, gs_before_diag>{});
  }
}

//! One work item (bundle, chunk) per workgroup: every chain of the bundle's
//! group on the bundle's slabs, the group's sum written to its slot (active
//! cells only).  Chunk entries are blocks of n^ND values (the slab digits,
//! the last fastest), one per other-index combination of the chunk; a
//! thread owns one block.  A resident item stages x, every factor table of
//! the group and both dimensions' lists once; otherwise a pass stages its
//! own table and list when they change.
template<typename P, int NT, int ND, int TPB>
__global__ void __launch_bounds__(TPB)
    gk_slab(gs_args a, const P *__restrict__ ctab, const gs_item *__restrict__ items,
            const P *__restrict__ x, P *work)
{
  extern __shared__ __align__(16) unsigned char gs_smem[];
  constexpr int nn = NT * NT;
  constexpr int ds = (ND == 1) ? NT : nn;
  const gs_item b = items[blockIdx.x];
  const int C = b.C;
  // a cell's blocks in LDS, padded by gs_pad values so that the blocks of
  // neighbouring cells fall on different LDS banks
  const int D = ds * C + gs_pad;
  const int BD = b.ncell * D;
  const int ntab_lds = b.resident ? b.ntab : 1;
  const int plane = b.tstride / ((nn + 1) / 2);
  gs_pass *pass = reinterpret_cast<gs_pass *>(gs_smem);
  P *X = reinterpret_cast<P *>(gs_smem + 16 * b.npass);
  P *Z = X + BD; // used when ND = 2
  P *tab = X + int64_t(BD) * ND;
  int *lists = reinterpret_cast<int *>(
      gs_smem + 16 * b.npass +
      ((int64_t(BD) * ND + int64_t(ntab_lds) * b.tstride) * int64_t(sizeof(P)) + 15) / 16 * 16);
  gs_copy<TPB>(reinterpret_cast<int *>(pass), reinterpret_cast<const int *>(a.passes + b.pass0),
               4 * b.npass);

  // this thread's block: cell c, other-index combination o of the chunk
  const int blk = threadIdx.x;
  const bool mine = blk < b.ncell * C;
  const int c = mine ? blk / C : 0;
  const int o = blk - (blk / C) * C;
  // where this entry's block starts within a cell, and its value (pair)
  // stride (pair-major, value-major or entry-major, as gs_at reads them);
  // cells are D values apart, D even for pair-major blocks (gs_pad is even),
  // so pairs stay 16-byte aligned
  const int vs = gs_pair_major<P, ds> ? 2 * C : (gs_value_major<P> ? C : 1);
  const int ob = gs_pair_major<P, ds> ? 2 * o : (gs_value_major<P> ? o : ds * o);
  const int gc = mine ? a.cells[b.cell0 + c] : -1;
  const bool active = gc >= 0 && gc < a.active_cells;
  const int64_t gbase = active ? int64_t(gc) * a.N + a.offs[b.off + o] : 0;
  auto gidx = [&](int si) -> int64_t {
    const int s0 = (ND == 1) ? si : si / NT;
    const int s1 = (ND == 1) ? 0 : si % NT;
    return gbase + int64_t(s0) * b.str[0] + ((ND == 1) ? 0 : int64_t(s1) * b.str[1]);
  };
  if (b.resident)
    gs_copy<TPB>(lists, a.lists + b.list0, b.llen[0] + (ND == 2 ? b.llen[1] : 0));
  P xv[ds];
#pragma unroll
  for (int si = 0; si < ds; si++)
    xv[si] = active ? x[gidx(si)] : P{0};
  if (b.resident)
    gs_copy<TPB>(tab, ctab + b.cb, b.ntab * b.tstride);
  if (mine)
  {
#pragma unroll
    for (int si = 0; si < ds; si++)
      X[c * D + gs_at<P, ds>(si, ob, vs)] = xv[si];
  }
  __syncthreads(); // the pass list is read before the first pass's barrier

  P acc[ds];
#pragma unroll
  for (int si = 0; si < ds; si++)
    acc[si] = 0;
  P next[ds];
#pragma unroll
  for (int si = 0; si < ds; si++)
    next[si] = 0;
  int cur_tab = -1, cur_j = -1;
  for (int pi = 0; pi < b.npass; pi++)
  {
    const gs_pass ps = pass[pi];
    if (!b.resident && (ps.tab != cur_tab || ps.j != cur_j))
    {
      // every earlier pass is done with the staged table and lists
      __syncthreads();
      if (ps.j != cur_j)
        gs_copy<TPB>(lists, a.lists + b.list0 + (ps.j == 0 ? 0 : b.llen[0]),
                     ps.j == 0 ? b.llen[0] : b.llen[1]);
      if (ps.tab != cur_tab)
        gs_copy<TPB>(tab, ctab + b.cb + int64_t(ps.tab) * b.tstride, b.tstride);
      cur_tab = ps.tab;
      cur_j = ps.j;
    }
    __syncthreads();
    if (mine)
    {
      const P *tb = b.resident ? tab + int64_t(ps.tab) * b.tstride : tab;
      const int *st = (b.resident && ps.j == 1) ? lists + b.llen[0] : lists;
      const int *dg = st + b.ncell + 1;
      const unsigned *ent = reinterpret_cast<const unsigned *>(dg + b.ncell);
      const P *in = (ps.mode >= 2) ? Z : X;
      P v[ds], w[ds];
#pragma unroll
      for (int si = 0; si < ds; si++)
        v[si] = w[si] = 0;
      if constexpr (ND == 2)
      {
        if (ps.mode == 3)
        {
          if (ps.j == 0)
            gs_pass_block<P, NT, ND, 0, 2>(in, X, tb, plane, st, dg, ent, c, ob, vs, ps.fill, v, w);
          else
            gs_pass_block<P, NT, ND, 1, 2>(in, X, tb, plane, st, dg, ent, c, ob, vs, ps.fill, v, w);
        }
        else if (ps.j == 1)
          gs_pass_block<P, NT, ND, 1, 1>(in, in, tb, plane, st, dg, ent, c, ob, vs, ps.fill, v, w);
        else
          gs_pass_block<P, NT, ND, 0, 1>(in, in, tb, plane, st, dg, ent, c, ob, vs, ps.fill, v, w);
      }
      else
        gs_pass_block<P, NT, ND, 0, 1>(in, in, tb, plane, st, dg, ent, c, ob, vs, ps.fill, v, w);
#pragma unroll
      for (int si = 0; si < ds; si++)
      {
        if (ps.mode == 1)
          Z[c * D + gs_at<P, ds>(si, ob, vs)] = v[si];
        else
          acc[si] += v[si];
        next[si] = w[si];
      }
    }
    if (ND == 2 && ps.mode == 3)
    {
      __syncthreads(); // the intermediate is read before it is replaced
      if (mine)
      {
#pragma unroll
        for (int si = 0; si < ds; si++)
          Z[c * D + gs_at<P, ds>(si, ob, vs)] = next[si];
      }
    }
    // the next pass may overwrite what this one read, or read what it wrote
    __syncthreads();
  }
  if (active)
  {
    P *out = work + int64_t(b.slot) * a.stride;
#pragma unroll
    for (int si = 0; si < ds; si++)
      out[gidx(si)] = acc[si];
  }
}

typedef int gs_int4 __attribute__((ext_vector_type(4)));

constexpr int gs_rec_steps = 8;                // connections per lane of a split item
constexpr int gs_rec_ints = 4 + gs_rec_steps;  // a lane record
//! 16-byte pieces of a factor table a thread reads ahead: 80 KB for 1024
//! threads, less where the blocks take the registers.
constexpr int gs_table_ahead(int n) { return n == 2 ? 5 : (n == 3 ? 2 : 1); }

//! First int of a lane record: its cell, the log2 of the lanes that share the
//! block, whether it is the first of them, and its connections.  The second
//! is the diagonal's list entry; from the fourth on the entries,
//! filled up by repeating one.
__host__ __device__ constexpr int gs_rec_meta(int c, int lg, bool first, int count)
{
  return c | lg << 10 | (first ? 1 : 0) << 13 | count << 16;
}

//! One split item (one chain of a large slab, one chunk) per workgroup: the
//! chain's one or two passes, its partial of every cell written out.  Blocks
//! in LDS as in gk_slab.
//! What bounded a thread per block here was waiting: for the longest list
//! (the level 0 and 1 cells are connected to their whole fibre, 128
//! connections at level 7, 10 on average), and for one read of memory after
//! another.  So a block with more than gs_rec_steps connections is shared by
//! 2, 4 ... 64 neighbouring lanes, whose sums meet by shuffles; every lane
//! reads its connections in one piece, a record ahead; and the factor table
//! of the second pass is read while the first one runs.  The 1248 items of
//! the d=6 n=2 level-7 FP64 Vlasov operator: 66 -> 48 us (LDS busy a third of
//! it; what is left is the way from one read of memory to the next at an
//! item's start, and two rounds of lanes where a pass has more than threads).
template<typename P, int NT, int ND, int TPB>
__global__ void __launch_bounds__(TPB, NT == 2 ? 4 : 1)
    gk_slab_chain(gs_args a, const P *__restrict__ ctab, const gs_item *__restrict__ items,
                  const P *__restrict__ x, P *part)
{
  extern __shared__ __align__(16) unsigned char gs_smem[];
  constexpr int ds = (ND == 1) ? NT : NT * NT;
  // the next connection's blocks are read ahead where registers allow
  constexpr bool ahead_blocks = (NT * NT + ds) * sizeof(P) <= 144 / (TPB / 512 > 1 ? 2 : 1);
  const gs_item b = items[blockIdx.x];
  const int C = b.C;
  const int D = ds * C + gs_pad;
  const int BD = b.ncell * D;
  P *X = reinterpret_cast<P *>(gs_smem);
  P *Z = X + BD; // used when ND = 2
  P *tab = reinterpret_cast<P *>(gs_smem + (int64_t(BD) * ND * sizeof(P) + 15) / 16 * 16);
  const int plane = b.tstride / ((NT * NT + 1) / 2);
  const int vs = gs_pair_major<P, ds> ? 2 * C : (gs_value_major<P> ? C : 1);
  auto base = [&](int o) {
    return gs_pair_major<P, ds> ? 2 * o : (gs_value_major<P> ? o : ds * o);
  };
  auto digit = [&](int si) { // entry si of a block, in its cell's tensor
    return (ND == 1) ? si * b.str[0] : si / NT * b.str[0] + si % NT * b.str[1];
  };
  // factor table of pass p, first pieces into registers
  const int pieces = b.tstride * int(sizeof(P)) / 16;
  constexpr int TA = gs_table_ahead(NT);
  gs_int4 ahead[TA];
  // a pass by value: an index into b would put b into scratch memory
  auto stage = [&](int p) { return p == 0 ? b.pass[0] : b.pass[1]; };
  auto table = [&](int p) {
    return reinterpret_cast<const gs_int4 *>(ctab + b.cb + int64_t(stage(p).ps.tab) * b.tstride);
  };
  auto read_table = [&](int p) {
    const gs_int4 *src = table(p); // past its end the last piece again
#pragma unroll
    for (int u = 0; u < TA; u++)
      ahead[u] = src[min(int(threadIdx.x) + u * TPB, pieces - 1)];
  };
  auto store_table = [&](int p) {
#pragma unroll
    for (int u = 0; u < TA; u++)
    {
      const int k = threadIdx.x + u * TPB;
      if (k < pieces)
        reinterpret_cast<gs_int4 *>(tab)[k] = ahead[u];
    }
    for (int k = threadIdx.x + TA * TPB; k < pieces; k += TPB)
      reinterpret_cast<gs_int4 *>(tab)[k] = table(p)[k];
  };
  // lane i of pass p: record and entry
  struct lane_rec
  {
    int o, off;
    gs_int4 head, e0, e1;
  };
  auto read_lane = [&](int p, int i) {
    lane_rec r;
    const gs_lane_pass q = stage(p);
    const int h = (i < q.nslot) ? a.slots[q.slot0 + i] : -1;
    r.o = h < 0 ? -1 : h >> 16;
    if (h >= 0)
    {
      const gs_int4 *rec =
          reinterpret_cast<const gs_int4 *>(a.recs + q.rec0 + (h & 0xffff) * gs_rec_ints);
      r.head = rec[0];
      r.e0 = rec[1];
      r.e1 = rec[2];
      r.off = a.offs[b.off + r.o];
    }
    return r;
  };
  read_table(0);
  lane_rec lane = read_lane(0, threadIdx.x);
  {
    const int c = threadIdx.x / C, o = threadIdx.x - c * C;
    const int gc = (c < b.ncell) ? a.cells[b.cell0 + c] : -1;
    const bool active = gc >= 0 && gc < a.active_cells;
    const int64_t gbase = active ? int64_t(gc) * a.N + a.offs[b.off + o] : 0;
    P xv[ds];
#pragma unroll
    for (int si = 0; si < ds; si++)
      xv[si] = active ? x[gbase + digit(si)] : P{0};
    store_table(0);
    if (c < b.ncell)
    {
#pragma unroll
      for (int si = 0; si < ds; si++)
        X[c * D + gs_at<P, ds>(si, base(o), vs)] = xv[si];
    }
  }
  __syncthreads();
  for (int p = 0; p < b.npass; p++)
  {
    const gs_pass ps = stage(p).ps;
    const int nslot = stage(p).nslot;
    const P *in = (ps.mode == 2) ? Z : X;
    if (p + 1 < b.npass)
      read_table(p + 1);
    // whole wavefronts: nslot is a multiple of 64, the most shared first
    for (int i = threadIdx.x; i < nslot; i += TPB)
    {
      const lane_rec r = lane;
      lane = read_lane(p, i + TPB);
      const int meta = (r.o < 0) ? 0 : r.head.x;
      const int c = meta & 1023, lg = meta >> 10 & 7, count = meta >> 16;
      const bool first = (meta >> 13 & 1) != 0;
      P v[ds];
#pragma unroll
      for (int si = 0; si < ds; si++)
        v[si] = 0;
      if (r.o >= 0)
      {
        const int ob = base(r.o);
        auto fma_j = [&](auto cols, const P(&av)[NT * NT], const P(&xv)[ds]) {
          if (ND == 1 || ps.j == 0)
            gs_block_fma<P, NT, ND, 0, cols.value>(av, xv, v);
          else
            gs_block_fma<P, NT, ND, 1, cols.value>(av, xv, v);
        };
        P av[NT * NT], xv[ds];
        if (first && ps.fill == gk_upper)
        {
          gs_block_load<P, NT, ND>(tab, plane, in, r.head.y, ob, vs, av, xv);
          fma_j(std::integral_constant<int, gs_from_diag>{}, av, xv);
        }
        const unsigned e[gs_rec_steps + 1] = {
            unsigned(r.e0.x), unsigned(r.e0.y), unsigned(r.e0.z), unsigned(r.e0.w), unsigned(r.e1.x),
            unsigned(r.e1.y), unsigned(r.e1.z), unsigned(r.e1.w), unsigned(r.e1.w)};
        if constexpr (ahead_blocks)
          gs_block_load<P, NT, ND>(tab, plane, in, e[0], ob, vs, av, xv);
#pragma unroll
        for (int s = 0; s < gs_rec_steps; s++)
        {
          if (s >= count)
            break;
          if constexpr (ahead_blocks)
          {
            P an[NT * NT], xn[ds];
            gs_block_load<P, NT, ND>(tab, plane, in, e[s + 1], ob, vs, an, xn);
            fma_j(std::integral_constant<int, gs_all>{}, av, xv);
#pragma unroll
            for (int k = 0; k < NT * NT; k++)
              av[k] = an[k];
#pragma unroll
            for (int k = 0; k < ds; k++)
              xv[k] = xn[k];
          }
          else
          {
            gs_block_load<P, NT, ND>(tab, plane, in, e[s], ob, vs, av, xv);
            fma_j(std::integral_constant<int, gs_all>{}, av, xv);
          }
        }
        if (first && ps.fill == gk_lower)
        {
          gs_block_load<P, NT, ND>(tab, plane, in, r.head.y, ob, vs, av, xv);
          fma_j(std::integral_constant<int, gs_before_diag>{}, av, xv);
        }
      }
      const int most = __builtin_amdgcn_readfirstlane(lg);
      for (int k = 0; k < most; k++)
#pragma unroll
        for (int si = 0; si < ds; si++)
        {
          const P w = __shfl_xor(v[si], 1 << k);
          v[si] += (k < lg) ? w : P{0};
        }
      if (!first)
        continue;
      if (ps.mode == 1)
      {
#pragma unroll
        for (int si = 0; si < ds; si++)
          Z[c * D + gs_at<P, ds>(si, base(r.o), vs)] = v[si];
      }
      else
      {
        P *out = part + (int64_t(b.part) + int64_t(c) * b.nch + b.chain) * a.N + r.off;
#pragma unroll
        for (int si = 0; si < ds; si++)
          out[digit(si)] = v[si];
      }
    }
    if (p + 1 < b.npass)
    {
      // the next pass reads what this one wrote, with its own table
      lane = read_lane(p + 1, threadIdx.x);
      __syncthreads();
      store_table(p + 1);
      __syncthreads();
    }
  }
}

//! Where gk_sum finds the slab groups' sums of cells whose chains ran split:
//! psplit[g * active cells + cell] is the cell's first partial in part (-1:
//! the group's slot holds the sum), gnch[g] the group's chains; group g's
//! slot is gslot0 + g.
template<typename P>
struct gs_split_view
{
  const int *psplit = nullptr;
  const int *gnch = nullptr;
  const P *part = nullptr;
  int gslot0 = 0, ngroups = 0;
};

//! y = (alpha * sum of the sources + beta*y + gamma*xg) / (1 - jdt * pc) (no
//! division when pc is null).  The sources, in order: x (src < 0, a term of
//! identity factors) or work-buffer slot src (a chain's last stage in chain
//! order, or a slab group's sum at the place of the group's first chain; for
//! a cell whose group chains ran split, the sum of its chain partials in
//! chain order).
template<typename P>
__global__ void __launch_bounds__(gk_threads)
    gk_sum(gk_args a, const int *__restrict__ src, int nsrc, const P *__restrict__ x,
           const P *__restrict__ work, P alpha, P beta, P *y, P gamma, const P *xg,
           const double *pc, double jdt, gs_split_view<P> sv)
{
  const int64_t dofs = a.active_cells * a.N;
  for (int64_t i = blockIdx.x * int64_t(gk_threads) + threadIdx.x; i < dofs;
       i += int64_t(gk_threads) * gridDim.x)
  {
    P sum = 0;
    const int64_t cell = (sv.psplit != nullptr) ? i / a.N : 0;
    const int64_t e = i - cell * a.N;
    for (int c = 0; c < nsrc; c++)
    {
      const int sl = src[c];
      const int gi = sl - sv.gslot0;
      const int pb = (sv.psplit != nullptr && gi >= 0 && gi < sv.ngroups)
                         ? sv.psplit[int64_t(gi) * a.active_cells + cell]
                         : -1;
      P v;
      if (sl < 0)
        v = x[i];
      else if (pb < 0)
        v = work[int64_t(sl) * a.stride + i];
      else
      {
        v = sv.part[int64_t(pb) * a.N + e];
        for (int k = 1; k < sv.gnch[gi]; k++)
          v += sv.part[(int64_t(pb) + k) * a.N + e];
      }
      sum += v;
    }
    P out = alpha * sum;
    if (beta != P{0})
      out += beta * y[i];
    if (gamma != P{0})
      out += gamma * xg[i];
    if (pc != nullptr)
      out = static_cast<P>(static_cast<double>(out) / (1.0 - jdt * pc[i]));
    y[i] = out;
  }
}

//! y = beta*y + gamma*xg (no terms), with the optional Jacobi division.
template<typename P>
__global__ void __launch_bounds__(gk_threads)
    gk_scale(int64_t dofs, P beta, P *y, P gamma, const P *xg, const double *pc, double jdt)
{
  for (int64_t i = blockIdx.x * int64_t(gk_threads) + threadIdx.x; i < dofs;
       i += int64_t(gk_threads) * gridDim.x)
  {
    P out = (beta != P{0}) ? beta * y[i] : P{0};
    if (gamma != P{0})
      out += gamma * xg[i];
    if (pc != nullptr)
      out = static_cast<P>(static_cast<double>(out) / (1.0 - jdt * pc[i]));
    y[i] = out;
  }
}

static int gk_blocks(int64_t work)
{
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((work + gk_threads - 1) /
                                                                     gk_threads,
                                                                 65536)));
}

//! gk_blocks rounded up to a multiple of the 8 XCDs (for gk_xcd_block).
static int gk_blocks_xcd(int64_t work)
{
  const int b = gk_blocks(work);
  return (b + 7) / 8 * 8;
}
} // namespace akm

//! Host and device data of a global operator.
struct akm_global_s
{
  using fibre_plan = akm::fibre_plan;
  using gk_lists = akm::gk_lists;
  int64_t active_cells = 0, cells = 0;
  std::vector<int> elem_host; // padded cells x d
  akm::dev_buffer<int> elem;
  akm::dev_buffer<int> nb_ptr[akm::gk_max_dims], nb_cell[akm::gk_max_dims],
      nb_q[akm::gk_max_dims], nb_diag[akm::gk_max_dims], order[akm::gk_max_dims];
  // chains: per chain its term, stages, and its stages' dimensions and fills
  // (gk_max_dims each), and its work-buffer slot
  struct
  {
    std::vector<int> term, nst, dim, fill, slot;
  } chains_host;
  akm::dev_buffer<int> ch_term, ch_nst, ch_dim, ch_fill, ch_slot;
  std::vector<akm::dev_buffer<int>> stage_list; // per stage: the chains that have it
  std::vector<int> stage_count;
  // first stage, cell layout: chains grouped by (dimension, fill), at most
  // gk_group_max per group
  akm::dev_buffer<int> first_ptr, first_chain;
  int first_groups = 0, first_largest = 0;
  bool first_grouped = false; // chosen by global_autotune
  bool xcd_order = false;     // chosen by global_autotune (cell layouts)
  int nchains = 0, nslots = 0, max_stages = 0;
  // chain layouts: 1 (a lane per DOF), 0 (a wavefront per cell, n^d <= 64),
  // or 8: the fibre walk, which has its own plan
  int lanes = 1;
  fibre_plan fl;
  std::vector<gk_lists> lists; // host fibre lists, per dimension
  std::vector<std::vector<int>> term_act; // non-identity dimensions per term
  int64_t fl_lanes = 0; // (lane, connection) steps of the fibre walk
  // the operator of a sparse-grid (pair) handle taken one dimension at a
  // time: no padding, no chain layouts, no Jacobi diagonal
  bool pair = false;
  bool slabs_built = false;
  // summation sources of gk_sum: chain layouts, and the slab layout
  akm::dev_buffer<int> src_chain, src_slab;
  int nsrc_chain = 0, nsrc_slab = 0;
  // slab layout (layout 6): groups of terms with the same one or two
  // non-identity dimensions, their bundles and work items; the other chains
  // run through the cell-layout stages
  bool slab = false; // chosen by global_autotune or akm_set_tuning
  int ngroups = 0;
  akm::dev_buffer<int> gs_passes, gs_tabs, gs_items, gs_cells, gs_lists, gs_offs, gs_qmap,
      gs_slots, gs_recs;
  // compact factor tables (per level bound, every group table), built from
  // vA by gs_tables with the layout and by every call that rewrites vA;
  // gs_lv: qmap starts then table starts per level bound (gs_levels + 1 each)
  akm::dev_buffer<unsigned char> gs_ctab;
  akm::dev_buffer<int> gs_lv;
  int64_t gs_ctab_count = 0;
  int gs_levels = 0;
  struct gs_launch
  {
    int tpb;     // 256 or 1024 threads
    int nd;      // slab dimensions of its groups
    bool split;  // one chain of a large slab per item
    bool side;   // on the side stream (split or 1024-thread items)
    int64_t lds; // dynamic LDS bytes (largest item of the launch)
    int first, count; // its items
  };
  std::vector<gs_launch> gs_launches;
  std::vector<int64_t> gs_item_lds; // dynamic LDS bytes per item
  // the last gs_moved items of the side launches run on the main stream after
  // its own launches (chosen by global_autotune: the stream that ends last
  // should be the main one, whose join then costs no wait)
  int gs_moved = 0;
  int gs_side_items = 0;
  // the 1024-thread launch (one large slab per workgroup, few workgroups)
  // runs beside the others on a stream of its own, forked and joined by events
  akm::dev_buffer<int> gs_psplit;     // per group and active cell: first partial or -1
  akm::dev_buffer<int> gs_gnch;       // per group: its chains
  akm::dev_buffer<unsigned char> gs_part; // split items' partials (N values each)
  hipStream_t gs_side = nullptr;
  hipEvent_t gs_fork = nullptr, gs_join = nullptr;
  ~akm_global_s()
  {
    if (gs_side)
      (void)hipStreamDestroy(gs_side);
    if (gs_fork)
      (void)hipEventDestroy(gs_fork);
    if (gs_join)
      (void)hipEventDestroy(gs_join);
  }
  std::vector<akm::dev_buffer<int>> stage_list_rest; // per stage: chains outside the groups
  std::vector<int> stage_count_rest;
  akm::dev_buffer<unsigned char> work;
  akm::dev_buffer<double> pc; // Jacobi diagonal (active DOFs)
  std::vector<int> c1_pntr_h, c1_indx_h, c1_diag_h;
  akm::dev_buffer<int> c1_diag; // device copy
  int64_t flops = 0;
};

namespace akm
{
void destroy_global(akm_global_s *g) { delete g; }

static gk_args global_args(akm_matrix_s const &m)
{
  const akm_global_s &g = *m.gk;
  gk_args a{};
  a.d = m.d;
  a.n = m.n;
  a.N = static_cast<int>(m.N);
  a.T = m.T;
  a.active_cells = g.active_cells;
  a.cells = g.cells;
  a.elem = g.elem.data();
  for (int k = 0; k < m.d; k++)
  {
    a.nb_ptr[k] = g.nb_ptr[k].data();
    a.nb_cell[k] = g.nb_cell[k].data();
    a.nb_q[k] = g.nb_q[k].data();
    a.nb_diag[k] = g.nb_diag[k].data();
    a.order[k] = g.order[k].data();
  }
  a.ch_term = g.ch_term.data();
  a.ch_nst = g.ch_nst.data();
  a.ch_dim = g.ch_dim.data();
  a.ch_fill = g.ch_fill.data();
  a.ch_slot = g.ch_slot.data();
  a.nchains = g.nchains;
  a.nslots = g.nslots;
  a.stride = g.cells * m.N;
  a.xcd_order = g.xcd_order;
  return a;
}

//! Launches one slab work-item class: `count` items from `items`, split ones
//! into the partials, the others into the work buffer.
template<typename P, int TPB>
static int gs_launch_class(hipStream_t stream, int n, int nd, bool split, gs_args const &ga,
                           const P *ctab, const gs_item *items, int count, int64_t lds,
                           const P *x, P *out)
{
  auto go = [&](auto kern) -> int {
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(lds)) != hipSuccess)
    {
      (void)hipGetLastError();
      return set_error(AKM_ERR_HIP, "global kron slab: %lld bytes of LDS refused",
                       static_cast<long long>(lds));
    }
    kern<<<count, TPB, static_cast<size_t>(lds), stream>>>(ga, ctab, items, x, out);
    return check_launch("global kron slab");
  };
  switch (n * 4 + nd)
  {
  case 2 * 4 + 1:
    return split ? go(gk_slab_chain<P, 2, 1, TPB>) : go(gk_slab<P, 2, 1, TPB>);
  case 2 * 4 + 2:
    return split ? go(gk_slab_chain<P, 2, 2, TPB>) : go(gk_slab<P, 2, 2, TPB>);
  case 3 * 4 + 1:
    return split ? go(gk_slab_chain<P, 3, 1, TPB>) : go(gk_slab<P, 3, 1, TPB>);
  case 3 * 4 + 2:
    return split ? go(gk_slab_chain<P, 3, 2, TPB>) : go(gk_slab<P, 3, 2, TPB>);
  case 4 * 4 + 1:
    return split ? go(gk_slab_chain<P, 4, 1, TPB>) : go(gk_slab<P, 4, 1, TPB>);
  case 4 * 4 + 2:
    return split ? go(gk_slab_chain<P, 4, 2, TPB>) : go(gk_slab<P, 4, 2, TPB>);
  default:
    return set_error(AKM_ERR_UNSUPPORTED, "global kron slab: n = %d", n);
  }
}

//! Compact factor tables: entry w of block qc of group table t at level
//! bound Lp is entry w of block qmap[qm0[Lp] + qc] of the (term, dimension)
//! tabs[t] of vA.  lv: qm0 (levels + 1 entries), then the table starts
//! cbase (levels + 1 entries).
template<typename P>
__global__ void __launch_bounds__(gk_threads)
    gs_tables(const P *__restrict__ vA, const int *__restrict__ tabs, int ntab,
              const int *__restrict__ qmap, const int *__restrict__ lv, int levels, int nn,
              int64_t tstride, int64_t cstride, int64_t count, P *ctab)
{
  for (int64_t i = blockIdx.x * int64_t(gk_threads) + threadIdx.x; i < count;
       i += int64_t(gk_threads) * gridDim.x)
  {
    int Lp = 0;
    while (Lp + 1 < levels && i >= lv[levels + 1 + Lp + 1])
      Lp++;
    const int64_t rem = i - lv[levels + 1 + Lp];
    const int nq = lv[Lp + 1] - lv[Lp];
    const int64_t per = gs_table_values(nq, nn);
    const int t = static_cast<int>(rem / per);
    const int r2 = static_cast<int>(rem - t * per);
    if (r2 >= nq * nn)
    {
      ctab[i] = P{0};
      continue;
    }
    // block qc, value w (gs_table_at)
    const bool planes = sizeof(P) == 8 && nn % 2 == 0;
    const int qc = planes ? r2 / 2 % nq : r2 / nn;
    const int w = planes ? r2 / 2 / nq * 2 + r2 % 2 : r2 - qc * nn;
    const int q = qmap[lv[Lp] + qc];
    ctab[i] = vA[int64_t(q) * cstride + int64_t(tabs[2 * t]) * tstride +
                 int64_t(tabs[2 * t + 1]) * nn + w];
  }
}

//! The compact factor tables of the slab layout, from vA.
template<typename P>
static int gs_refresh(akm_matrix_s const &m, akm_global_s &g)
{
  const int nn = m.n * m.n;
  const int64_t tstride = int64_t(m.d) * nn;
  gs_tables<P><<<gk_blocks(g.gs_ctab_count), gk_threads, 0, m.stream>>>(
      reinterpret_cast<const P *>(m.vA.data()), g.gs_tabs.data(),
      static_cast<int>(g.gs_tabs.size() / 2), g.gs_qmap.data(), g.gs_lv.data(), g.gs_levels, nn,
      tstride, tstride * m.T, g.gs_ctab_count, reinterpret_cast<P *>(g.gs_ctab.data()));
  return check_launch("global kron slab tables");
}

static int gs_refresh(akm_matrix_s const &m, akm_global_s &g)
{
  return (m.prec == AKM_F64) ? gs_refresh<double>(m, g) : gs_refresh<float>(m, g);
}

int global_tables(akm_matrix_s &m)
{
  akm_global_s &g = *m.gk;
  if (g.fl.built)
    AKM_TRY(fibre_refresh(m, g.fl, m.stream));
  if (g.ngroups > 0)
    AKM_TRY(gs_refresh(m, g));
  return AKM_SUCCESS;
}

//! Every slab group's sum into its work-buffer slot.
template<typename P>
static int gs_apply(akm_matrix_s &m, const P *x, P *work)
{
  akm_global_s &g = *m.gk;
  gs_args ga{};
  ga.d = m.d;
  ga.n = m.n;
  ga.N = static_cast<int>(m.N);
  ga.T = m.T;
  ga.active_cells = g.active_cells;
  ga.stride = g.cells * m.N;
  ga.passes = reinterpret_cast<const gs_pass *>(g.gs_passes.data());
  ga.cells = g.gs_cells.data();
  ga.lists = g.gs_lists.data();
  ga.offs = g.gs_offs.data();
  ga.slots = g.gs_slots.data();
  ga.recs = g.gs_recs.data();
  const P *ctab = reinterpret_cast<const P *>(g.gs_ctab.data());
  // the side launches come first and run on the side stream; gk_sum
  // follows the join
  // with every side item moved there is nothing to fork
  const bool fork = g.gs_side != nullptr && g.gs_moved < g.gs_side_items;
  if (fork)
  {
    AKM_HIP(hipEventRecord(g.gs_fork, m.stream));
    AKM_HIP(hipStreamWaitEvent(g.gs_side, g.gs_fork, 0));
  }
  const hipStream_t side = fork ? g.gs_side : m.stream;
  // items [0, bound) of the side launches run on the side stream, the rest
  // after the main stream's own launches
  const int bound = fork ? g.gs_side_items - std::min(g.gs_moved, g.gs_side_items)
                         : g.gs_side_items;
  P *part = reinterpret_cast<P *>(g.gs_part.data());
  auto run = [&](hipStream_t s, auto const &l, int first, int count) -> int {
    if (count <= 0)
      return AKM_SUCCESS;
    const gs_item *items = reinterpret_cast<const gs_item *>(g.gs_items.data()) + first;
    const int64_t lds = *std::max_element(g.gs_item_lds.begin() + first,
                                          g.gs_item_lds.begin() + first + count);
    P *out = l.split ? part : work;
    if (l.tpb == 1024)
      return gs_launch_class<P, 1024>(s, m.n, l.nd, l.split, ga, ctab, items, count, lds, x, out);
    if (l.tpb == 512)
      return gs_launch_class<P, 512>(s, m.n, l.nd, l.split, ga, ctab, items, count, lds, x, out);
    return gs_launch_class<P, 256>(s, m.n, l.nd, l.split, ga, ctab, items, count, lds, x, out);
  };
  for (auto const &l : g.gs_launches)
    if (l.side)
      AKM_TRY(run(side, l, l.first, std::min(l.first + l.count, bound) - l.first));
  for (auto const &l : g.gs_launches)
    if (!l.side)
      AKM_TRY(run(m.stream, l, l.first, l.count));
  for (auto const &l : g.gs_launches)
    if (l.side)
    {
      const int f = std::max(l.first, bound);
      AKM_TRY(run(m.stream, l, f, l.first + l.count - f));
    }
  if (fork)
  {
    AKM_HIP(hipEventRecord(g.gs_join, g.gs_side));
    AKM_HIP(hipStreamWaitEvent(m.stream, g.gs_join, 0));
  }
  return AKM_SUCCESS;
}

template<typename P>
static int global_apply_typed(akm_matrix_s &m, P alpha, const P *x, P beta, P *y, P gamma,
                              const P *xg, bool jacobi, double jdt)
{
  akm_global_s &g = *m.gk;
  const int64_t dofs = g.active_cells * m.N;
  const double *pc = jacobi ? g.pc.data() : nullptr;
  if (g.nchains == 0 || alpha == P{0} || dofs == 0)
  {
    if (dofs > 0)
      gk_scale<P><<<gk_blocks(dofs), gk_threads, 0, m.stream>>>(dofs, beta, y, gamma, xg, pc,
                                                                  jdt);
    return check_launch("global kron scale");
  }
  // the walk's last stage writes y while other workgroups still read x: a
  // global handle's apply in place takes the chain layout, which forms y in a
  // pass of its own that reads x at its own positions only
  const bool in_place = !g.pair && x < y + dofs && y < x + dofs;
  if (!g.slab && g.lanes == 8 && !in_place)
    return fibre_apply<P>(m, g.fl, alpha, x, beta, y, gamma, xg, pc, jdt);
  const gk_args a = global_args(m);
  const P *vA = reinterpret_cast<const P *>(m.vA.data());
  P *work = reinterpret_cast<P *>(g.work.data());
  // the slab layout runs the chains outside its groups in the cell layout
  const bool slab = g.slab;
  const int lanes = (slab || g.lanes == 8) ? (m.N <= wave_size ? 0 : 1) : g.lanes;
  for (int st = 0; st < g.max_stages; st++)
  {
    const int nl = slab ? g.stage_count_rest[st] : g.stage_count[st];
    if (nl == 0)
      continue;
    const int *list = slab ? g.stage_list_rest[st].data() : g.stage_list[st].data();
    const int blocks = (lanes == 0) ? gk_blocks_xcd(g.cells * nl * wave_size)
                                    : gk_blocks(g.cells * m.N * nl);
    if (!slab && lanes == 0 && st == 0 && g.first_grouped && g.first_largest > 1 && m.n >= 2 &&
        m.n <= 4)
    {
      // chains sharing their first-stage input read it once
      const int fb = gk_blocks_xcd(g.cells * g.first_groups * wave_size);
      const int *gp = g.first_ptr.data(), *gc = g.first_chain.data();
      const int ng = g.first_groups;
      const bool two = g.first_largest <= 2;
      if (m.n == 2 && two)
        gk_cell_first<P, 2, 2><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
      else if (m.n == 2)
        gk_cell_first<P, 2, 4><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
      else if (m.n == 3 && two)
        gk_cell_first<P, 3, 2><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
      else if (m.n == 3)
        gk_cell_first<P, 3, 4><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
      else if (two)
        gk_cell_first<P, 4, 2><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
      else
        gk_cell_first<P, 4, 4><<<fb, gk_threads, 0, m.stream>>>(a, vA, gp, gc, ng, x, work);
    }
    else if (lanes == 0)
    {
      switch (m.n)
      {
      case 2:
        gk_cell_stage<P, 2><<<blocks, gk_threads, 0, m.stream>>>(a, vA, list, nl, st, x, work);
        break;
      case 3:
        gk_cell_stage<P, 3><<<blocks, gk_threads, 0, m.stream>>>(a, vA, list, nl, st, x, work);
        break;
      case 4:
        gk_cell_stage<P, 4><<<blocks, gk_threads, 0, m.stream>>>(a, vA, list, nl, st, x, work);
        break;
      default:
        gk_cell_stage<P, 0><<<blocks, gk_threads, 0, m.stream>>>(a, vA, list, nl, st, x, work);
      }
    }
    else
      gk_stage<P><<<blocks, gk_threads, 0, m.stream>>>(a, vA, list, nl, st, x, work);
    AKM_TRY(check_launch("global kron stage"));
  }
  if (slab)
    AKM_TRY(gs_apply<P>(m, x, work));
  const int *src = slab ? g.src_slab.data() : g.src_chain.data();
  const int nsrc = slab ? g.nsrc_slab : g.nsrc_chain;
  gs_split_view<P> sv{};
  if (slab && g.gs_psplit.size() > 0)
  {
    sv.psplit = g.gs_psplit.data();
    sv.gnch = g.gs_gnch.data();
    sv.part = reinterpret_cast<const P *>(g.gs_part.data());
    sv.gslot0 = 2 * g.nslots;
    sv.ngroups = g.ngroups;
  }
  gk_sum<P><<<gk_blocks(dofs), gk_threads, 0, m.stream>>>(a, src, nsrc, x, work, alpha, beta, y,
                                                          gamma, xg, pc, jdt, sv);
  return check_launch("global kron sum");
}

int global_apply(akm_matrix_s &m, double alpha, const void *x, double beta, void *y,
                 double gamma, const void *xg, bool jacobi, double jdt)
{
  if (m.prec == AKM_F64)
    return global_apply_typed<double>(m, alpha, static_cast<const double *>(x), beta,
                                      static_cast<double *>(y), gamma,
                                      static_cast<const double *>(xg), jacobi, jdt);
  return global_apply_typed<float>(m, static_cast<float>(alpha), static_cast<const float *>(x),
                                   static_cast<float>(beta), static_cast<float *>(y),
                                   static_cast<float>(gamma), static_cast<const float *>(xg),
                                   jacobi, jdt);
}

bool apply_f32_between(akm_matrix_s &m, const double *v, double c, double *w)
{
  if (m.prec != AKM_F32 || !m.gk || (m.mode != mode_global && (!m.factored || m.pair_kernels || m.pair_tuned)))
    return false;
  akm_global_s &g = *m.gk;
  if (g.slab || g.lanes != 8 || g.active_cells == 0)
    return false;
  std::lock_guard<std::mutex> lock(m.factored_mtx);
  return fibre_apply_between(m, g.fl, v, c, w);
}

int global_update(akm_matrix_s &m, const void *vA)
{
  AKM_HIP(hipMemcpyAsync(m.vA.data(), vA, m.num_vA * m.esize, hipMemcpyHostToDevice, m.stream));
  AKM_TRY(global_device_jacobi(m));
  AKM_TRY(global_tables(m));
  AKM_HIP(hipStreamSynchronize(m.stream));
  return AKM_SUCCESS;
}

//! The Jacobi diagonal of the reference's implicit step
//! (build_preconditioner, src/asgard_kronmult_matrix.cpp:1016-1067): for
//! every active DOF, the sum over terms of the product over dimensions of the
//! 1D factors' diagonal entries (every dimension, identity factors included),
//! one thread per DOF, products and sums rounded one by one (no contraction
//! into fma).
template<typename P>
__global__ void __launch_bounds__(gk_threads)
    gk_jacobi(int64_t active_cells, int d, int n, int T, int64_t N, const int *elem,
              const int *c1_diag, const P *vA, double *pc)
{
  const int64_t nn = int64_t(n) * n;
  for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < active_cells * N;
       idx += int64_t(gridDim.x) * blockDim.x)
  {
    const int64_t c = idx / N, e = idx - c * N;
    double sum = 0;
    for (int t = 0; t < T; t++)
    {
      double prod = 1;
      int64_t rest = e;
      for (int k = d - 1; k >= 0; k--)
      {
        const int s = static_cast<int>(rest % n);
        rest /= n;
        const int64_t q = c1_diag[elem[c * d + k]];
        prod = __dmul_rn(prod, static_cast<double>(vA[((q * T + t) * d + k) * nn + s * n + s]));
      }
      sum = __dadd_rn(sum, prod);
    }
    pc[idx] = sum;
  }
}

int global_device_jacobi(akm_matrix_s &m)
{
  akm_global_s &g = *m.gk;
  if (g.c1_diag.size() == 0)
    AKM_TRY(g.c1_diag.upload(g.c1_diag_h.data(), int64_t(g.c1_diag_h.size()), m.stream));
  const int64_t work = g.active_cells * m.N;
  if (work == 0)
    return AKM_SUCCESS;
  AKM_TRY(g.pc.allocate(work));
  if (m.prec == AKM_F64)
    gk_jacobi<double><<<gk_blocks(work), gk_threads, 0, m.stream>>>(
        g.active_cells, m.d, m.n, m.T, m.N, g.elem.data(), g.c1_diag.data(),
        reinterpret_cast<const double *>(m.vA.data()), g.pc.data());
  else
    gk_jacobi<float><<<gk_blocks(work), gk_threads, 0, m.stream>>>(
        g.active_cells, m.d, m.n, m.T, m.N, g.elem.data(), g.c1_diag.data(),
        reinterpret_cast<const float *>(m.vA.data()), g.pc.data());
  return check_launch("global kron Jacobi diagonal");
}

//! Builds the fibre-walk plan and its tables on first use.
static int need_fibre_plan(akm_matrix_s &m)
{
  akm_global_s &g = *m.gk;
  if (g.fl.built)
    return AKM_SUCCESS;
  g.fl = fibre_plan();
  AKM_TRY(build_fibre_plan(m, g.active_cells, g.cells, g.elem_host.data(), g.lists, g.term_act,
                           g.c1_diag_h, g.fl));
  AKM_TRY(fibre_refresh(m, g.fl, m.stream));
  AKM_HIP(hipStreamSynchronize(m.stream)); // another stream may be captured next
  return AKM_SUCCESS;
}

bool factored_batch_plan(akm_matrix_s const &m, fibre_plan &plan, int &rc)
{
  rc = AKM_SUCCESS;
  // (the batch kernel's forms: n = 3 alone past 64 entries a cell)
  if (!m.factored || m.pair_kernels || !m.gk || m.prec != AKM_F64 || m.gk->max_stages > 1 || m.n < 2 || m.n > 4 ||
      m.N > (m.n == 3 ? 1024 : 64))
    return false;
  akm_global_s const &g = *m.gk;
  rc = build_fibre_plan(m, g.active_cells, g.cells, g.elem_host.data(), g.lists, g.term_act,
                        g.c1_diag_h, plan);
  return rc == AKM_SUCCESS;
}

int64_t global_flops(akm_matrix_s const &m) { return m.gk ? m.gk->flops : 0; }

int global_layout(akm_matrix_s const &m)
{
  if (!m.gk)
    return 0;
  if (m.gk->slab)
    return 6;
  if (m.gk->lanes == 0)
    return (m.gk->first_grouped ? 3 : 2) + (m.gk->xcd_order ? 2 : 0);
  return m.gk->lanes;
}

int global_stages(akm_matrix_s const &m) { return m.gk ? m.gk->max_stages : 0; }

bool global_shares_work(akm_matrix_s const &m)
{
  // (a global handle's apply in place runs in the chain layout)
  return m.gk && (!m.gk->pair || m.gk->slab || m.gk->fl.vectors > 0);
}

int global_set_layout(akm_matrix_s &m, int layout)
{
  if (!m.gk)
    return set_error(AKM_ERR_INVALID, "not a global kron matrix");
  if (layout == 0)
    return AKM_SUCCESS;
  if (layout != 1 && layout != 8 && (layout < 2 || layout > 6))
    return set_error(AKM_ERR_INVALID, "global kron layout %d is not 1, 2, 3, 4, 5, 6 or 8",
                     layout);
  const bool cell = (layout >= 2 && layout <= 5);
  if (cell && m.N > wave_size)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: the cell layout needs n^d <= 64");
  if (layout == 8)
    AKM_TRY(need_fibre_plan(m));
  m.gk->slab = (layout == 6);
  if (m.gk->slab)
  {
    m.gk->lanes = 0;
    m.gk->first_grouped = false;
    m.gk->xcd_order = false;
    return AKM_SUCCESS;
  }
  m.gk->lanes = cell ? 0 : layout;
  m.gk->first_grouped = (layout == 3 || layout == 5);
  m.gk->xcd_order = (layout == 4 || layout == 5);
  return AKM_SUCCESS;
}

//! Fibre walks of up to this many (lane, connection) steps are planned
//! without being asked for (their slot records take about half as many
//! bytes).
constexpr int64_t fl_lanes_tuned = int64_t(1) << 26;
//! The layout of a handle that is not tuned: the fibre walk up to this many
//! (lane, connection) steps, then the slab layout where it takes every chain.
//! With two dimensions a term the slabs save the walk's way of the
//! intermediate through memory; us per apply of walk / slabs on the d = 6
//! n = 2 Vlasov operator: 6.0 M steps (level 5) FP64 37 / 43, FP32 29 / 39;
//! 22 M (level 6) 87 / 44 and 70 / 45; 76 M (level 7) 254 / 100.  With one
//! dimension a term neither is ahead throughout: d = 6 n = 2 7.4 M 29 / 23,
//! 25 M 85 / 101; d = 4 n = 2 level 8 4.3 M 15 / 56; d = 5 n = 3 4.3 M 34 / 17.
static int64_t fl_lanes_default(int stages)
{
  return (stages > 1) ? int64_t(1) << 23 : int64_t(1) << 26;
}

//! Up to this many steps the fibre walk is always the faster of the two.
constexpr int64_t fl_lanes_small = int64_t(1) << 20;

//! The layout used until akm_autotune or akm_set_tuning picks one; -1 when an
//! operator of a pair handle has none.
static int default_layout(akm_matrix_s const &m, akm_global_s const &g)
{
  if (g.fl_lanes <= fl_lanes_default(g.max_stages))
    return 8;
  if (g.ngroups > 0 && (g.max_stages == 0 || g.stage_count_rest[0] == 0))
    return 6;
  if (g.fl_lanes <= fl_lanes_tuned)
    return 8;
  if (g.pair)
    return -1;
  return (m.N <= wave_size) ? 2 : 1;
}

static int need_slabs(akm_matrix_s &m, akm_global_s &g);

//! Times the row layouts on the operator itself (y is overwritten) and
//! keeps the fastest.
int global_autotune(akm_matrix_s &m, const void *x, void *y, double &best_ms)
{
  akm_global_s &g = *m.gk;
  hipEvent_t e0, e1;
  AKM_HIP(hipEventCreate(&e0));
  AKM_HIP(hipEventCreate(&e1));
  float best = -1;
  // (the layout so far, should no candidate run)
  int best_lanes = g.lanes;
  bool best_grouped = g.first_grouped;
  int rc = AKM_SUCCESS;
  bool best_xcd = g.xcd_order, best_slab = g.slab;
  int best_moved = g.gs_moved;
  // layouts 1 and 8 (when its records stay small), then the cell layout with
  // and without the grouped first stage (shared input reads against fewer, longer wavefronts), each
  // cell layout with and without the XCD-contiguous workgroup order, then
  // the slab layout (when some term has one or two non-identity dimensions)
  // with 0-100 % of its side-stream items moved to the main stream (100:
  // one stream, no fork and join)
  const int shapes[7][4] = {{1, 0, 0, 0}, {8, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 1, 0},
                            {0, 1, 0, 0}, {0, 1, 1, 0}, {0, 0, 0, 1}};
  for (auto const &shape : shapes)
  {
    const int lanes = shape[0];
    const bool grouped = shape[1] != 0;
    const bool xcd = shape[2] != 0;
    const bool slab = shape[3] != 0;
    if (lanes == 0 && !slab && m.N > wave_size)
      continue;
    if (grouped && g.first_largest < 2)
      continue;
    if (g.pair && lanes != 8 && !slab)
      continue;
    // (without room for the slabs the walk is left)
    if (slab && g.pair && g.fl_lanes > fl_lanes_small && need_slabs(m, g) != AKM_SUCCESS)
      (void)hipGetLastError();
    if (slab && g.ngroups == 0)
      continue;
    if (lanes == 8)
    {
      if (g.fl_lanes > fl_lanes_tuned)
        continue;
      rc = need_fibre_plan(m);
      if (rc != AKM_SUCCESS)
        break;
    }
    g.lanes = lanes;
    g.first_grouped = grouped;
    g.xcd_order = xcd;
    g.slab = slab;
    const int percents[9] = {0, 10, 20, 30, 40, 50, 65, 80, 100};
    const int nmoves = (slab && g.gs_side != nullptr) ? 9 : 1;
    for (int mi = 0; mi < nmoves && rc == AKM_SUCCESS; mi++)
    {
      g.gs_moved = g.gs_side_items * percents[mi] / 100;
      rc = global_apply(m, 1.0, x, 0.0, y, 0.0, nullptr, false, 0.0);
      if (rc != AKM_SUCCESS)
        break;
      (void)hipEventRecord(e0, m.stream);
      for (int r = 0; r < 5 && rc == AKM_SUCCESS; r++)
        rc = global_apply(m, 1.0, x, 0.0, y, 0.0, nullptr, false, 0.0);
      (void)hipEventRecord(e1, m.stream);
      float ms = 0;
      if (rc == AKM_SUCCESS && hipEventSynchronize(e1) == hipSuccess &&
          hipEventElapsedTime(&ms, e0, e1) == hipSuccess && (best < 0 || ms < best))
      {
        best = ms;
        best_lanes = lanes;
        best_grouped = grouped;
        best_xcd = xcd;
        best_slab = slab;
        best_moved = g.gs_moved;
      }
    }
    if (rc != AKM_SUCCESS)
      break;
  }
  g.lanes = best_lanes;
  g.first_grouped = best_grouped;
  g.xcd_order = best_xcd;
  g.slab = best_slab;
  g.gs_moved = best_moved;
  best_ms = (best < 0) ? 1e300 : best / 5;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

int factored_shape(akm_matrix_s const &m) { return global_layout(m) + 16 * m.gk->gs_moved; }

int factored_set_shape(akm_matrix_s &m, int shape)
{
  int layout = shape % 16;
  if (layout == 6 && need_slabs(m, *m.gk) != AKM_SUCCESS)
    (void)hipGetLastError();
  // the number may come from another grid of the same size, or there is no
  // room for the slabs
  if (layout == 6 && m.gk->ngroups == 0)
    layout = 8;
  AKM_TRY(global_set_layout(m, layout));
  m.gk->gs_moved = shape / 16;
  return AKM_SUCCESS;
}

//! Ancestors of a 1D cell in the volume hierarchy: its parent chain down to
//! cell 0 (the part of a connect_1d volume row before the diagonal,
//! src/asgard_grid_1d.hpp:159-260).
static void parents_1d(int i, std::vector<int> &out)
{
  out.clear();
  while (i > 0)
  {
    i = (i == 1) ? 0 : i / 2;
    out.push_back(i);
  }
}

//! Level of a 1D cell index (0 for cell 0, l for 2^(l-1) <= i < 2^l).
static int level_1d(int i)
{
  int l = 0;
  while (i > 0)
  {
    i >>= 1;
    l++;
  }
  return l;
}

//! One bundle while the slab plan is made.
struct gs_plan_bundle
{
  std::vector<int> cells;
  int C = 1, Lp = 0, tpb = 256;
};

//! Where the lanes of a split bundle's pass are: slots, records.
struct gs_lane_range
{
  int slot0 = -1, nslot = 0, rec0 = 0;
};

//! The lanes of a pass over a split bundle's cells with the `fill` part of
//! their lists: every block shared by as many lanes (a power of two, at most
//! 64) as its list has lots of gs_rec_steps connections, lane k taking every
//! lanes-th from the k-th on; the most shared first, so that a block's lanes
//! stay in one wavefront; filled up with -1 to whole wavefronts.  entry(p) is
//! the packed LDS offsets of list position p; false when something does not
//! fit.
template<typename Entry>
static bool gs_lanes(std::vector<int> const &cells, gk_lists const &ls, int fill, int C,
                     Entry &&entry, std::vector<int> &slots, std::vector<int> &recs)
{
  std::vector<int> by_lg[7];
  auto range = [&](int gc) {
    return std::make_pair(fill == gk_upper ? ls.diag[gc] + 1 : ls.ptr[gc],
                          fill == gk_lower ? ls.diag[gc] : ls.ptr[gc + 1]);
  };
  for (size_t c = 0; c < cells.size(); c++)
  {
    auto const [lo, hi] = range(cells[c]);
    int lg = 0;
    while (lg < 6 && (gs_rec_steps << lg) < static_cast<int>(hi - lo))
      lg++;
    if ((gs_rec_steps << lg) < static_cast<int>(hi - lo))
      return false; // more than 512 connections: its table does not fit LDS either
    by_lg[lg].push_back(static_cast<int>(c));
  }
  int nrec = 0;
  for (int lg = 6; lg >= 0; lg--)
    for (int c : by_lg[lg])
    {
      auto const [lo, hi] = range(cells[c]);
      const int lanes = 1 << lg;
      unsigned diag = 0;
      if (!entry(ls.diag[cells[c]], diag))
        return false;
      for (int sub = 0; sub < lanes; sub++)
      {
        const int count = std::max<int>(0, static_cast<int>(hi - lo) - sub + lanes - 1) / lanes;
        recs.insert(recs.end(), {gs_rec_meta(c, lg, sub == 0, count), static_cast<int>(diag), 0, 0});
        unsigned e = diag;
        for (int k = 0; k < gs_rec_steps; k++)
        {
          if (k < count && !entry(lo + sub + k * lanes, e))
            return false;
          recs.push_back(static_cast<int>(e));
        }
      }
      for (int o = 0; o < C; o++)
        for (int sub = 0; sub < lanes; sub++)
          slots.push_back((nrec + sub) | o << 16);
      nrec += lanes;
    }
  while (slots.size() % wave_size != 0)
    slots.push_back(-1);
  return nrec <= 0x10000;
}

//! Builds the slab layout: groups of the terms with one or two non-identity
//! dimensions (act[t] after the flux swap), their slabs, bundles, lists and
//! work items.  A group whose largest slab does not fit one workgroup at
//! one other-index combination per chunk is left to the cell-layout stages.
static int build_slabs(akm_matrix_s &m, akm_global_s &g)
{
  std::vector<gk_lists> const &lists = g.lists;
  std::vector<std::vector<int>> const &term_act = g.term_act;
  std::vector<int> const &ch_term = g.chains_host.term, &ch_nst = g.chains_host.nst,
                         &ch_dim = g.chains_host.dim, &ch_fill = g.chains_host.fill,
                         &ch_slot = g.chains_host.slot;
  const int d = m.d, n = m.n, T = m.T;
  const int L = m.max_level;
  const int nn = n * n;
  const int esize = static_cast<int>(m.esize);
  // compact factor index per level bound Lp: connect_1d entries with row and
  // column below 2^Lp, in connect_1d order
  std::vector<std::vector<int>> qc_of(L + 1);
  std::vector<int> qmap, qm0;
  for (int Lp = 0; Lp <= L; Lp++)
  {
    qm0.push_back(static_cast<int>(qmap.size()));
    qc_of[Lp].assign(g.c1_indx_h.size(), -1);
    const int lim = 1 << Lp;
    int cnt = 0;
    for (int r = 0; r < lim && r + 1 < static_cast<int>(g.c1_pntr_h.size()); r++)
      for (int q = g.c1_pntr_h[r]; q < g.c1_pntr_h[r + 1]; q++)
        if (g.c1_indx_h[q] < lim)
        {
          qc_of[Lp][q] = cnt++;
          qmap.push_back(q);
        }
  }
  qm0.push_back(static_cast<int>(qmap.size()));

  // groups by the set of non-identity dimensions
  std::vector<int> term_group(T, -1);
  std::vector<std::vector<int>> gdims;
  for (int t = 0; t < T; t++)
  {
    const int na = static_cast<int>(term_act[t].size());
    if (na < 1 || na > 2)
      continue;
    std::vector<int> key = term_act[t];
    std::sort(key.begin(), key.end());
    size_t gi = 0;
    while (gi < gdims.size() && gdims[gi] != key)
      gi++;
    if (gi == gdims.size())
      gdims.push_back(key);
    term_group[t] = static_cast<int>(gi);
  }

  std::vector<gs_bundle> bundles;
  std::vector<gs_group> groups;
  std::vector<int> passes, tabs, items, cells, lists_img, offs, slots, recs;
  struct item_rec
  {
    int bundle, h, tpb, nd;
    int64_t lds;
    int resident;
    int chain = -1;          // >= 0: this chain of the group only (a split item)
    int Lp = 0;              // level bound of its bundle
    int pass_off = 0, pass_cnt = 0; // its passes within the group's
    gs_pass pass[2] = {};
    gs_lane_range lanes[2]; // its passes' lanes
  };
  std::vector<item_rec> irec;
  // a group's plan, its positions counted from its own first ones
  struct group_plan
  {
    bool kept = false;
    gs_group rec{};
    std::vector<gs_bundle> bundles;
    std::vector<int> cells, lists, slots, recs, offs, tabs, passes;
    std::vector<item_rec> items;
  };
  std::vector<group_plan> plans(gdims.size());
  std::vector<int> loc(g.cells, -1);
  auto plan_group = [&](size_t gi, group_plan &gp) {
    for (int attempt = 0; attempt < 2 && !gp.kept; attempt++)
  {
    // small bundles of gs_blocks_small_first blocks, else (second attempt,
    // when those do not fit) of gs_blocks_small; a failed attempt commits
    // nothing
    const int blocks_small = (attempt == 0) ? gs_blocks_small_first(esize) : gs_blocks_small;
    if (attempt == 1 && blocks_small == gs_blocks_small_first(esize))
      break;
    const std::vector<int> &S = gdims[gi];
    const int nd = static_cast<int>(S.size());
    const int ds = (nd == 1) ? n : nn;
    const int64_t gs_cap_small = int64_t(blocks_small) * ds; // values
    const int64_t gs_cap_large = int64_t(gs_blocks_large) * ds;
    if (n < 2 || n > 4)
      continue; // the slab kernels hold n^nd-value blocks in registers
    int call = 1;
    for (int k = nd; k < d; k++)
      call *= n;
    // slabs: cells equal in every 1D index outside S, cell order kept
    // (slabs in the order of those indices)
    std::vector<int> other, by_slab;
    for (int k = 0; k < d; k++)
      if (std::find(S.begin(), S.end(), k) == S.end())
        other.push_back(k);
    order_by_dims(d, g.cells, g.elem_host.data(), other, m.M, by_slab);
    int group_chains = 0;
    for (size_t c = 0; c < ch_term.size(); c++)
      if (term_group[ch_term[c]] == static_cast<int>(gi))
        group_chains++;
    // bundles: small slabs packed up to gs_cap_small values, a larger slab
    // alone with its other-index combinations split into chunks
    std::vector<gs_plan_bundle> plan;
    bool ok = true;
    gs_plan_bundle open;
    open.tpb = blocks_small;
    int64_t open_vals = 0;
    auto slab_level = [&](std::vector<int> const &sc) {
      int lp = 0;
      for (int c : sc)
        for (int k : S)
          lp = std::max(lp, level_1d(g.elem_host[int64_t(c) * d + k]));
      return lp;
    };
    std::vector<int> sc;
    for (int64_t s0 = 0; s0 < g.cells;)
    {
      sc.clear();
      for (; s0 < g.cells; s0++)
      {
        const int c = by_slab[s0];
        bool same = true;
        for (int k : other)
          same = same && (sc.empty() || g.elem_host[int64_t(c) * d + k] ==
                                            g.elem_host[int64_t(sc[0]) * d + k]);
        if (!same)
          break;
        sc.push_back(c);
      }
      const int64_t msz = static_cast<int64_t>(sc.size());
      const int64_t full = msz * ds * call;
      const int lp = slab_level(sc);
      if (full <= gs_cap_small)
      {
        if (open_vals + full > gs_cap_small)
        {
          plan.push_back(open);
          open = gs_plan_bundle();
          open.tpb = blocks_small;
          open_vals = 0;
        }
        open.cells.insert(open.cells.end(), sc.begin(), sc.end());
        open.C = call;
        open.Lp = std::max(open.Lp, lp);
        open_vals += full;
        continue;
      }
      if (lp >= gs_split_level && group_chains > 1)
      {
        // its chains run split: chunks for 512 threads that let two
        // workgroups share a CU, else for 1024 (d=6 n=2 Vlasov, levels 5 / 6 /
        // 7: 31 / 39 / 92 us; 256 threads first 30 / 45 / 101, 1024 only
        // 32 / 60 / 89)
        const int nq = qm0[lp + 1] - qm0[lp];
        gs_plan_bundle one;
        one.cells = sc;
        one.Lp = lp;
        for (int tpb : {512, 1024})
        {
          one.tpb = tpb;
          one.C = call;
          auto fits = [&] {
            return msz * one.C <= tpb &&
                   gs_split_lds(esize, nd, n, static_cast<int>(msz), one.C, nq) <=
                       (tpb == 512 ? gs_lds_max / 2 : gs_lds_max);
          };
          while (one.C > 1 && !fits())
            one.C /= n;
          ok = fits();
          if (ok)
            break;
        }
        if (!ok)
          break;
        plan.push_back(one);
        continue;
      }
      const int64_t cap = (msz * ds <= gs_cap_small) ? gs_cap_small : gs_cap_large;
      if (msz * ds > cap)
      {
        ok = false;
        break;
      }
      gs_plan_bundle one;
      one.cells = sc;
      one.Lp = lp;
      one.tpb = (cap == gs_cap_small) ? blocks_small : 1024;
      one.C = call;
      while (msz * ds * one.C > cap)
        one.C /= n;
      plan.push_back(one);
    }
    if (ok && !open.cells.empty())
      plan.push_back(open);
    if (!ok)
      continue;

    // the group's terms in chain order: factor tables (term, S[j]) at
    // term index * nd + j
    std::vector<int> gterms;
    for (size_t c = 0; c < ch_term.size(); c++)
      if (term_group[ch_term[c]] == static_cast<int>(gi) &&
          std::find(gterms.begin(), gterms.end(), ch_term[c]) == gterms.end())
        gterms.push_back(ch_term[c]);
    const int ntab = static_cast<int>(gterms.size()) * nd;
    int npass = 0;
    std::vector<std::pair<int, int>> gchains; // (first pass, passes) per chain
    std::vector<gs_pass> gpass;               // their passes
    std::vector<int> own;                     // the group's chains
    auto pass_of = [&](int c, int st) {
      const int ti = static_cast<int>(std::find(gterms.begin(), gterms.end(), ch_term[c]) -
                                      gterms.begin());
      const int j = (ch_dim[c * gk_max_dims + st] == S[0]) ? 0 : 1;
      return gs_pass{ti * nd + j, j, ch_fill[c * gk_max_dims + st],
                     (ch_nst[c] == 1) ? 0 : (st == 0 ? 1 : 2)};
    };
    auto add_pass = [](std::vector<int> &to, gs_pass const &ps) {
      to.insert(to.end(), {ps.tab, ps.j, ps.fill, ps.mode});
    };
    // the first stage of chain c is the last of chain c2 of the same term:
    // they run at once and share the lists and factor blocks (d=6 n=2 Vlasov
    // at level 5 33.5 -> 31 us, level 6 43 -> 39 us, level 7 the same)
    auto merged = [&](int c, int c2) {
      return nd == 2 && ch_term[c] == ch_term[c2] && ch_nst[c] == 2 && ch_nst[c2] == 2 &&
             ch_dim[c * gk_max_dims] == ch_dim[c2 * gk_max_dims + 1] &&
             ch_fill[c * gk_max_dims] == ch_fill[c2 * gk_max_dims + 1];
    };
    for (size_t c = 0; c < ch_term.size(); c++)
      if (term_group[ch_term[c]] == static_cast<int>(gi))
      {
        own.push_back(static_cast<int>(c));
        gchains.emplace_back(npass, ch_nst[c]);
        npass += ch_nst[c];
        for (int st = 0; st < ch_nst[c]; st++)
          gpass.push_back(pass_of(static_cast<int>(c), st));
      }

    // each bundle's cells by their longest list, longest first: a wavefront
    // walks as many connections as its longest list, so long lists share
    // wavefronts (the order changes no operation order within a value)
    for (auto &pb : plan)
    {
      auto longest = [&](int gc) {
        int len = 0;
        for (int k : S)
          len = std::max(len, lists[k].ptr[gc + 1] - lists[k].ptr[gc]);
        return len;
      };
      std::vector<std::pair<int, int>> by_length; // (-length, cell)
      by_length.reserve(pb.cells.size());
      for (int c : pb.cells)
        by_length.emplace_back(-longest(c), c);
      std::stable_sort(by_length.begin(), by_length.end(),
                       [](auto const &u, auto const &v) { return u.first < v.first; });
      for (size_t c = 0; c < pb.cells.size(); c++)
        pb.cells[c] = by_length[c].second;
    }

    // lists, LDS sizes and items of the plan (checked before anything is kept)
    std::vector<gs_bundle> b_rec;
    std::vector<int> p_cells, p_lists, p_slots, p_recs;
    std::vector<item_rec> p_items;
    for (size_t bi = 0; bi < plan.size() && ok; bi++)
    {
      gs_plan_bundle const &pb = plan[bi];
      const int ncell = static_cast<int>(pb.cells.size());
      gs_bundle rec{};
      rec.cell0 = static_cast<int>(p_cells.size());
      rec.ncell = ncell;
      rec.C = pb.C;
      rec.Lp = pb.Lp;
      rec.list0 = static_cast<int>(p_lists.size());
      for (int c = 0; c < ncell; c++)
        loc[pb.cells[c]] = c;
      // element offset of the connected cell in x / the intermediate,
      // element offset of its factor block in the table; false outside the
      // slab (cannot happen) or past 16-bit offsets
      auto entry = [&](gk_lists const &ls, int64_t p, unsigned &e) {
        const int64_t xo = int64_t(loc[ls.cell[p]]) * (ds * pb.C + gs_pad);
        const int64_t ao = int64_t(qc_of[pb.Lp][ls.q[p]]) * ((esize == 8 && nn % 2 == 0) ? 2 : nn);
        e = static_cast<unsigned>(xo) | (static_cast<unsigned>(ao) << 16);
        return xo >= 0 && ao >= 0 && xo <= 0xffff && ao <= 0xffff;
      };
      // a slab with long connection lists (level bound >= gs_split_level) runs
      // one workgroup per chain: its passes are the longest.  The lanes of its
      // passes, by (slab dimension, fill)
      const bool split = pb.Lp >= gs_split_level && gchains.size() > 1;
      gs_lane_range lanes_of[2][3];
      for (size_t pi = 0; split && ok && pi < gpass.size(); pi++)
      {
        auto &where = lanes_of[gpass[pi].j][gpass[pi].fill];
        if (where.slot0 >= 0)
          continue;
        gk_lists const &ls = lists[S[gpass[pi].j]];
        const size_t s0 = p_slots.size();
        where.slot0 = static_cast<int>(s0);
        where.rec0 = static_cast<int>(p_recs.size());
        ok = gs_lanes(pb.cells, ls, gpass[pi].fill, pb.C,
                      [&](int64_t p, unsigned &e) { return entry(ls, p, e); }, p_slots, p_recs);
        where.nslot = static_cast<int>(p_slots.size() - s0);
      }
      int nent_max = 0, nent_sum = 0;
      for (int j = 0; j < nd && ok && !split; j++)
      {
        // image: ncell + 1 starts, ncell diagonal positions, the entries
        gk_lists const &ls = lists[S[j]];
        const size_t img = p_lists.size();
        p_lists.resize(img + 2 * size_t(ncell) + 1);
        int cnt = 0;
        for (int c = 0; c < ncell && ok; c++)
        {
          const int gc = pb.cells[c];
          p_lists[img + c] = cnt;
          p_lists[img + ncell + 1 + c] = cnt + ls.diag[gc] - ls.ptr[gc];
          for (int p = ls.ptr[gc]; p < ls.ptr[gc + 1]; p++)
          {
            unsigned e;
            if (!entry(ls, p, e))
            {
              ok = false;
              break;
            }
            p_lists.push_back(static_cast<int>(e));
            cnt++;
          }
        }
        p_lists[img + ncell] = cnt;
        rec.llen[j] = static_cast<int>(p_lists.size() - img);
        nent_max = std::max(nent_max, cnt);
        nent_sum += cnt;
      }
      for (int c = 0; c < ncell; c++)
        loc[pb.cells[c]] = -1;
      if (!ok)
        break;
      const int nq = qm0[pb.Lp + 1] - qm0[pb.Lp];
      // everything staged once when that keeps two workgroups per CU, else
      // one table and one list at a time
      int64_t lds = gs_lds_bytes(esize, nd, n, ncell, pb.C, nq, ntab,
                                 int64_t(nd) * (2 * ncell + 1) + nent_sum, npass);
      rec.resident = (lds <= gs_lds_resident) ? 1 : 0;
      if (!rec.resident)
        lds = gs_lds_bytes(esize, nd, n, ncell, pb.C, nq, 1, 2 * ncell + 1 + nent_max, npass);
      if (split)
        lds = gs_split_lds(esize, nd, n, ncell, pb.C, nq);
      if (lds > gs_lds_max)
      {
        ok = false;
        break;
      }
      b_rec.push_back(rec);
      p_cells.insert(p_cells.end(), pb.cells.begin(), pb.cells.end());
      for (int h = 0; h < call / pb.C; h++)
      {
        if (!split)
        {
          p_items.push_back({static_cast<int>(bi), h, pb.tpb, nd, lds, rec.resident});
          continue;
        }
        for (size_t k = 0; k < gchains.size(); k++)
        {
          item_rec r{static_cast<int>(bi), h, pb.tpb, nd, lds, 0};
          r.chain = static_cast<int>(k);
          r.Lp = pb.Lp;
          r.pass_off = gchains[k].first;
          r.pass_cnt = gchains[k].second;
          for (int st = 0; st < r.pass_cnt; st++)
          {
            auto const &ps = gpass[r.pass_off + st];
            r.pass[st] = ps;
            r.lanes[st] = lanes_of[ps.j][ps.fill];
          }
          p_items.push_back(r);
        }
      }
    }
    if (!ok)
      continue;
    // the group is kept
    gs_group &grec = gp.rec;
    grec.nd = nd;
    for (int j = 0; j < nd; j++)
    {
      grec.dim[j] = S[j];
      int str = 1;
      for (int k = S[j] + 1; k < d; k++)
        str *= n;
      grec.str[j] = str;
    }
    grec.call = call;
    for (int o = 0; o < call; o++)
    {
      // digits of o over the other dimensions, the last one fastest
      int rem = o, off = 0, str = 1;
      for (int k = d - 1; k >= 0; k--)
      {
        if (std::find(S.begin(), S.end(), k) == S.end())
        {
          off += (rem % n) * str;
          rem /= n;
        }
        str *= n;
      }
      gp.offs.push_back(off);
    }
    grec.ntab = ntab;
    for (int t : gterms)
      for (int j = 0; j < nd; j++)
        gp.tabs.insert(gp.tabs.end(), {t, S[j]});
    for (size_t c = 0; c < own.size(); c++)
    {
      if (c + 1 < own.size() && merged(own[c], own[c + 1]))
      {
        // F then L and U then F: U, both F at once, L
        gs_pass f = pass_of(own[c], 0);
        f.mode = 3;
        add_pass(gp.passes, pass_of(own[c + 1], 0));
        add_pass(gp.passes, f);
        add_pass(gp.passes, pass_of(own[c], 1));
        c++;
        continue;
      }
      for (int st = 0; st < ch_nst[own[c]]; st++)
        add_pass(gp.passes, pass_of(own[c], st));
    }
    grec.npass = static_cast<int>(gp.passes.size() / 4);
    gp.bundles = std::move(b_rec);
    gp.cells = std::move(p_cells);
    gp.lists = std::move(p_lists);
    gp.slots = std::move(p_slots);
    gp.recs = std::move(p_recs);
    gp.items = std::move(p_items);
    gp.kept = true;
  }
  };
  for (size_t gi = 0; gi < gdims.size(); gi++)
    plan_group(gi, plans[gi]);
  // the kept groups one after another
  std::vector<int> gslot(gdims.size(), -1);
  int ngroups = 0;
  auto append = [](auto &to, auto const &from) { to.insert(to.end(), from.begin(), from.end()); };
  for (size_t gi = 0; gi < gdims.size(); gi++)
  {
    group_plan &gp = plans[gi];
    if (!gp.kept)
      continue;
    gp.rec.off0 = static_cast<int>(offs.size());
    gp.rec.tab0 = static_cast<int>(tabs.size() / 2);
    gp.rec.pass0 = static_cast<int>(passes.size() / 4);
    gp.rec.slot = 2 * g.nslots + ngroups;
    const int bundle0 = static_cast<int>(bundles.size()), cell0 = static_cast<int>(cells.size()),
              list0 = static_cast<int>(lists_img.size()), slot0 = static_cast<int>(slots.size()),
              rec0 = static_cast<int>(recs.size());
    for (auto &b : gp.bundles)
    {
      b.group = ngroups;
      b.cell0 += cell0;
      b.list0 += list0;
    }
    for (auto &r : gp.items)
    {
      r.bundle += bundle0;
      for (auto &l : r.lanes)
        if (l.slot0 >= 0)
        {
          l.slot0 += slot0;
          l.rec0 += rec0;
        }
    }
    groups.push_back(gp.rec);
    append(bundles, gp.bundles);
    append(cells, gp.cells);
    append(lists_img, gp.lists);
    append(slots, gp.slots);
    append(recs, gp.recs);
    append(offs, gp.offs);
    append(tabs, gp.tabs);
    append(passes, gp.passes);
    append(irec, gp.items);
    gslot[gi] = ngroups++;
    gp = group_plan();
  }
  for (int t = 0; t < T; t++)
    if (term_group[t] >= 0 && gslot[term_group[t]] < 0)
      term_group[t] = -1; // its group did not fit: cell-layout stages
  g.ngroups = ngroups;

  // launches: 1024-thread items, then the small bundles' (512 or 256
  // threads), per slab dimension count (one launch for all items of a size,
  // largest LDS first, measured faster than separate launches above and
  // below 32 KB of LDS)
  // the side stream takes the 1024-thread items (the split items of the
  // largest slabs among them), about half the work on the Vlasov operator;
  // they come first, and gs_apply may run the last gs_moved of them on the
  // main stream
  auto on_side = [](item_rec const &r) { return r.chain >= 0 || r.tpb == 1024; };
  auto cls = [&](item_rec const &r) {
    const int side = on_side(r) ? 0 : 1;
    const int size = (r.tpb == 1024) ? 0 : (r.tpb == 512 ? 1 : 2);
    return ((side * 3 + size) * 2 + (r.nd - 1)) * 2 + (r.chain >= 0 ? 0 : 1);
  };
  // within a launch the largest items first (the longest-running workgroups
  // start early)
  std::vector<uint64_t> keys; // class, then LDS bytes (below 2^20) falling
  for (auto const &r : irec)
    keys.push_back(static_cast<uint64_t>(cls(r)) << 20 |
                   static_cast<uint64_t>((1 << 20) - 1 - r.lds));
  std::vector<int> item_order;
  radix_order(keys, 26, item_order);
  std::vector<item_rec> sorted;
  sorted.reserve(irec.size());
  for (int i : item_order)
    sorted.push_back(irec[i]);
  irec.swap(sorted);
  g.gs_launches.clear();
  g.gs_item_lds.clear();
  g.gs_side_items = 0;
  // partials of split bundles: per bundle ncell * chains of N values
  const size_t nbundles = bundles.size();
  std::vector<int64_t> part0(nbundles, -1);
  std::vector<int> nch_of(nbundles, 0);
  int64_t nparts = 0;
  for (auto const &r : irec)
    if (r.chain >= 0)
      nch_of[r.bundle] = std::max(nch_of[r.bundle], r.chain + 1);
  for (size_t bi = 0; bi < nbundles; bi++)
    if (nch_of[bi] > 0)
    {
      part0[bi] = nparts;
      nparts += int64_t(bundles[bi].ncell) *
                nch_of[bi];
    }
  if (nparts > (int64_t(1) << 31) - 1)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: too many slab partials");
  // compact factor tables, per level bound every group table: cbase[Lp]
  const int64_t ntab_all = static_cast<int64_t>(tabs.size() / 2);
  std::vector<int64_t> cbase(L + 2, 0);
  for (int Lp = 0; Lp <= L; Lp++)
    cbase[Lp + 1] = cbase[Lp] + ntab_all * gs_table_values(qm0[Lp + 1] - qm0[Lp], nn);
  if (cbase[L + 1] > (int64_t(1) << 31) - 1)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: slab factor tables too large");
  const gs_bundle *hb = bundles.data();
  const gs_group *hg = groups.data();
  for (size_t i = 0; i < irec.size(); i++)
  {
    const gs_bundle &bb = hb[irec[i].bundle];
    const gs_group &gg = hg[bb.group];
    gs_item it{};
    it.cell0 = bb.cell0;
    it.ncell = bb.ncell;
    it.C = bb.C;
    it.tstride = gs_table_values(qm0[bb.Lp + 1] - qm0[bb.Lp], nn);
    it.cb = static_cast<int>(cbase[bb.Lp] + int64_t(gg.tab0) * it.tstride);
    it.resident = irec[i].resident;
    it.list0 = bb.list0;
    it.llen[0] = bb.llen[0];
    it.llen[1] = bb.llen[1];
    it.nd = gg.nd;
    it.str[0] = gg.str[0];
    it.str[1] = gg.str[1];
    it.off = gg.off0 + irec[i].h * bb.C;
    it.ntab = gg.ntab;
    const bool split = irec[i].chain >= 0;
    it.pass0 = gg.pass0;
    it.npass = split ? irec[i].pass_cnt : gg.npass;
    // a split item writes its chain's partials, which gk_sum adds
    it.slot = gg.slot;
    it.part = split ? part0[irec[i].bundle] : -1;
    it.nch = split ? nch_of[irec[i].bundle] : 0;
    it.chain = split ? irec[i].chain : 0;
    for (int st = 0; split && st < irec[i].pass_cnt; st++)
    {
      it.pass[st] = gs_lane_pass{irec[i].pass[st], irec[i].lanes[st].slot0,
                                 irec[i].lanes[st].nslot, irec[i].lanes[st].rec0};
    }
    const int *ip = reinterpret_cast<const int *>(&it);
    items.insert(items.end(), ip, ip + sizeof(gs_item) / sizeof(int));
    if (g.gs_launches.empty() || cls(irec[i - 1]) != cls(irec[i]))
      g.gs_launches.push_back({irec[i].tpb, irec[i].nd, split, on_side(irec[i]), 0,
                               static_cast<int>(i), 0});
    auto &l = g.gs_launches.back();
    l.lds = std::max(l.lds, irec[i].lds);
    l.count++;
    g.gs_item_lds.push_back(irec[i].lds);
    if (on_side(irec[i]))
      g.gs_side_items = static_cast<int>(i) + 1;
  }
  // until global_autotune measures it, a quarter of the side items run on
  // the main stream (near the best split of the FP64 Vlasov operator)
  g.gs_moved = g.gs_side_items / 4;
  // gk_sum's view of split bundles (every chunk of a split bundle is split):
  // per group and active cell the first of its chain partials
  if (nparts > 0)
  {
    std::vector<int> psplit(size_t(ngroups) * g.active_cells, -1), gnch(ngroups, 0);
    for (size_t bi = 0; bi < nbundles; bi++)
    {
      if (nch_of[bi] == 0)
        continue;
      const gs_bundle &bb = hb[bi];
      gnch[bb.group] = nch_of[bi];
      for (int c = 0; c < bb.ncell; c++)
      {
        const int gc = cells[bb.cell0 + c];
        if (gc < g.active_cells)
          psplit[size_t(bb.group) * g.active_cells + gc] =
              static_cast<int>(part0[bi] + int64_t(c) * nch_of[bi]);
      }
    }
    AKM_TRY(g.gs_psplit.upload(psplit.data(), int64_t(psplit.size())));
    AKM_TRY(g.gs_gnch.upload(gnch.data(), int64_t(gnch.size())));
  }
  if (nparts > 0)
    AKM_TRY(g.gs_part.allocate(nparts * m.N * esize));
  if (!g.gs_launches.empty() && g.gs_launches[0].side && !g.gs_launches.back().side &&
      g.gs_side == nullptr)
  {
    AKM_HIP(hipStreamCreateWithFlags(&g.gs_side, hipStreamNonBlocking));
    AKM_HIP(hipEventCreateWithFlags(&g.gs_fork, hipEventDisableTiming));
    AKM_HIP(hipEventCreateWithFlags(&g.gs_join, hipEventDisableTiming));
  }
  if (ngroups > 0)
  {
    AKM_TRY(g.gs_passes.upload(passes.data(), int64_t(passes.size())));
    AKM_TRY(g.gs_tabs.upload(tabs.data(), int64_t(tabs.size())));
    AKM_TRY(g.gs_items.upload(items.data(), int64_t(items.size())));
    AKM_TRY(g.gs_cells.upload(cells.data(), int64_t(cells.size())));
    AKM_TRY(g.gs_lists.upload(lists_img.data(), int64_t(lists_img.size())));
    AKM_TRY(g.gs_offs.upload(offs.data(), int64_t(offs.size())));
    if (!slots.empty())
    {
      AKM_TRY(g.gs_slots.upload(slots.data(), int64_t(slots.size())));
      AKM_TRY(g.gs_recs.upload(recs.data(), int64_t(recs.size())));
    }
    AKM_TRY(g.gs_qmap.upload(qmap.data(), int64_t(qmap.size())));
    std::vector<int> lv(qm0.begin(), qm0.end());
    for (int64_t v : cbase)
      lv.push_back(static_cast<int>(v));
    AKM_TRY(g.gs_lv.upload(lv.data(), int64_t(lv.size())));
    AKM_TRY(g.gs_ctab.allocate(cbase[L + 1] * esize));
    g.gs_ctab_count = cbase[L + 1];
    g.gs_levels = L + 1;
  }

  // the chains outside the groups, per stage, and the summation sources
  g.stage_list_rest.clear();
  g.stage_list_rest.resize(g.max_stages);
  g.stage_count_rest.assign(g.max_stages, 0);
  for (int st = 0; st < g.max_stages; st++)
  {
    std::vector<int> list;
    for (size_t c = 0; c < ch_term.size(); c++)
      if (term_group[ch_term[c]] < 0 && ch_nst[c] >= st + 1)
        list.push_back(static_cast<int>(c));
    g.stage_count_rest[st] = static_cast<int>(list.size());
    if (!list.empty())
      AKM_TRY(g.stage_list_rest[st].upload(list.data(), int64_t(list.size())));
  }
  std::vector<int> src_chain, src_slab;
  std::vector<bool> emitted(gdims.size(), false);
  for (size_t c = 0; c < ch_term.size(); c++)
  {
    const int ns = ch_nst[c];
    const int own = (ns == 0) ? -1 : ((ns - 1) & 1) * g.nslots + ch_slot[c];
    src_chain.push_back(own);
    const int gi = term_group[ch_term[c]];
    if (gi < 0)
      src_slab.push_back(own);
    else if (!emitted[gi])
    {
      emitted[gi] = true;
      src_slab.push_back(2 * g.nslots + gslot[gi]);
    }
  }
  g.nsrc_chain = static_cast<int>(src_chain.size());
  g.nsrc_slab = static_cast<int>(src_slab.size());
  if (!src_chain.empty())
    AKM_TRY(g.src_chain.upload(src_chain.data(), int64_t(src_chain.size())));
  if (!src_slab.empty())
    AKM_TRY(g.src_slab.upload(src_slab.data(), int64_t(src_slab.size())));
  return AKM_SUCCESS;
}

//! Builds the slab layout and its tables on first use.  Chains outside its groups run in the
//! chain layouts, which a pair handle does not have.
static int need_slabs(akm_matrix_s &m, akm_global_s &g)
{
  if (g.slabs_built)
    return AKM_SUCCESS;
  g.slabs_built = true;
  auto build = [&]() -> int {
    AKM_TRY(build_slabs(m, g));
    if (g.pair && g.max_stages > 0 && g.stage_count_rest[0] > 0)
      g.ngroups = 0;
    if (g.ngroups == 0)
      return AKM_SUCCESS;
    if (g.pair)
      AKM_TRY(g.work.allocate(int64_t(g.ngroups) * g.cells * m.N * int64_t(m.esize)));
    AKM_TRY(gs_refresh(m, g));
    AKM_HIP(hipStreamSynchronize(m.stream)); // another stream may be captured next
    return AKM_SUCCESS;
  };
  const int rc = build();
  if (rc != AKM_SUCCESS)
    g.ngroups = 0; // too large, or out of memory: what was made is not used
  return rc;
}

//! Builds the padded cell set, the fibres, the chains and the work buffers
//! (make_global_kron_matrix, src/asgard_kronmult_matrix.cpp:1198-1334).  With
//! `pair` (the operator of a sparse-grid handle, whose cells need no padding)
//! only what the fibre walk and the slab layout use.  `repeated` = the first
//! cell that equals an earlier one (nothing is built then), or -1.  Its
//! layout is the caller's to set with `pair`, else the default one.
static int build_global(akm_matrix_s &m, const std::vector<int> &elem_active,
                        const int *active_mask, const int *flux_dim, bool pair,
                        int64_t &repeated)
{
  auto g = std::unique_ptr<akm_global_s, void (*)(akm_global_s *)>(new akm_global_s(),
                                                                    destroy_global);
  const int d = m.d;
  const int64_t nact = m.rows;
  g->active_cells = nact;
  g->pair = pair;
  g->elem_host = elem_active;
  repeated = -1;

  // ancestry completion (compute_ancestry_completion over the volume
  // hierarchy, src/asgard_indexset.cpp:243-318): add the missing ancestors
  // in every dimension until none is missing; padding sorted.  A grid of
  // whole levels misses none.
  if (!pair && !whole_level_grid(d, nact, elem_active.data()))
  {
    std::map<std::vector<int>, int64_t> index;
    std::vector<int> key(d), anc;
    for (int64_t c = 0; c < nact; c++)
    {
      key.assign(elem_active.begin() + c * d, elem_active.begin() + (c + 1) * d);
      index.emplace(key, c);
    }
    std::vector<std::vector<int>> frontier;
    for (int64_t c = 0; c < nact; c++)
      frontier.emplace_back(elem_active.begin() + c * d, elem_active.begin() + (c + 1) * d);
    std::map<std::vector<int>, int> padset;
    while (!frontier.empty())
    {
      std::vector<std::vector<int>> next;
      for (auto const &cell : frontier)
        for (int k = 0; k < d; k++)
        {
          parents_1d(cell[k], anc);
          for (int a : anc)
          {
            key = cell;
            key[k] = a;
            if (index.count(key) == 0 && padset.count(key) == 0)
            {
              padset.emplace(key, 0);
              next.push_back(key);
            }
          }
        }
      frontier.swap(next);
    }
    for (auto const &kv : padset)
      g->elem_host.insert(g->elem_host.end(), kv.first.begin(), kv.first.end());
  }
  g->cells = static_cast<int64_t>(g->elem_host.size() / d);
  if (g->cells * m.N > (int64_t(1) << 40))
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: too many padded DOFs");

  // connect_1d (full hierarchy), the pattern of every 1D factor
  if (pair)
  {
    g->c1_pntr_h = m.conn_pntr_host;
    g->c1_indx_h = m.conn_indx_host;
    g->c1_diag_h = m.conn_diag_host;
  }
  else
    AKM_TRY(build_connect_1d(m.max_level, true, g->c1_pntr_h, g->c1_indx_h, g->c1_diag_h));

  // per dimension: the fibres (cells equal in every other 1D index) and for
  // every cell its connected cells of the fibre, 1D index ascending
  std::vector<int64_t> nnz_dim(d, 0); // DOF-level pattern entries per dimension
  g->lists.resize(d);
  std::vector<gk_lists> &lists = g->lists;
  for (int k = 0; k < d; k++)
  {
    std::vector<int> ord;
    AKM_TRY(build_fibre_lists(d, g->cells, g->elem_host.data(), k, m.M, g->c1_pntr_h,
                              g->c1_indx_h, g->c1_diag_h, lists[k], ord, repeated));
    if (repeated >= 0)
      return AKM_SUCCESS;
    nnz_dim[k] = static_cast<int64_t>(lists[k].cell.size()) * m.n * m.N;
    if (pair)
      continue;
    AKM_TRY(g->nb_ptr[k].upload(lists[k].ptr.data(), int64_t(lists[k].ptr.size())));
    AKM_TRY(g->nb_cell[k].upload(lists[k].cell.data(), int64_t(lists[k].cell.size())));
    AKM_TRY(g->nb_q[k].upload(lists[k].q.data(), int64_t(lists[k].q.size())));
    AKM_TRY(g->nb_diag[k].upload(lists[k].diag.data(), int64_t(lists[k].diag.size())));
    // processing order: fibre by fibre
    AKM_TRY(g->order[k].upload(ord.data(), int64_t(ord.size())));
  }
  if (!pair)
    AKM_TRY(g->elem.upload(g->elem_host.data(), int64_t(g->elem_host.size())));

  // chains (kronmult::permutes, src/device/asgard_kronmult.hpp:152-220, and
  // the active-direction order of src/asgard_kronmult_matrix.cpp:1313-1331)
  auto &[ch_term, ch_nst, ch_dim, ch_fill, ch_slot] = g->chains_host;
  std::vector<std::vector<int>> &term_act = g->term_act;
  term_act.resize(m.T);
  for (int t = 0; t < m.T; t++)
  {
    std::vector<int> act;
    for (int k = 0; k < d; k++)
      if (active_mask == nullptr || active_mask[t * d + k] != 0)
        act.push_back(k);
    const int na = static_cast<int>(act.size());
    if (na > 1 && flux_dim != nullptr)
    {
      // the reference swaps positions 0 and flux_dim of the active list
      const int fd = flux_dim[t];
      if (fd >= 0 && fd < na && fd != act[0])
        std::swap(act[0], act[fd]);
    }
    term_act[t] = act;
    if (na == 0)
    {
      ch_term.push_back(t);
      ch_nst.push_back(0);
      ch_dim.insert(ch_dim.end(), gk_max_dims, 0);
      ch_fill.insert(ch_fill.end(), gk_max_dims, 0);
      continue;
    }
    for (int p = 0; p < (1 << (na - 1)); p++)
    {
      std::vector<int> sgn(1, 0);
      int bits = p;
      for (int dd = 1; dd < na; dd++)
      {
        sgn.push_back((bits % 2 == 0) ? dd : -dd);
        bits /= 2;
      }
      std::sort(sgn.begin(), sgn.end());
      ch_term.push_back(t);
      ch_nst.push_back(na);
      for (int st = 0; st < gk_max_dims; st++)
      {
        if (st < na)
        {
          ch_dim.push_back(act[std::abs(sgn[st])]);
          ch_fill.push_back(sgn[st] < 0 ? gk_upper : (sgn[st] > 0 ? gk_lower : gk_full));
        }
        else
        {
          ch_dim.push_back(0);
          ch_fill.push_back(0);
        }
      }
    }
  }
  g->nchains = static_cast<int>(ch_term.size());
  g->max_stages = 0;
  int nslots = 0;
  for (int c = 0; c < g->nchains; c++)
  {
    g->max_stages = std::max(g->max_stages, ch_nst[c]);
    ch_slot.push_back((ch_nst[c] >= 1 && !pair) ? nslots++ : -1);
  }
  g->nslots = nslots;
  if (g->nchains > 0 && !pair)
  {
    AKM_TRY(g->ch_term.upload(ch_term.data(), int64_t(ch_term.size())));
    AKM_TRY(g->ch_nst.upload(ch_nst.data(), int64_t(ch_nst.size())));
    AKM_TRY(g->ch_dim.upload(ch_dim.data(), int64_t(ch_dim.size())));
    AKM_TRY(g->ch_fill.upload(ch_fill.data(), int64_t(ch_fill.size())));
    AKM_TRY(g->ch_slot.upload(ch_slot.data(), int64_t(ch_slot.size())));
  }
  // chains per stage (those with more than st stages)
  g->stage_list.resize(g->max_stages);
  g->stage_count.assign(g->max_stages, 0);
  for (int st = 0; st < g->max_stages; st++)
  {
    std::vector<int> list;
    for (int c = 0; c < g->nchains; c++)
      if (ch_nst[c] >= st + 1)
        list.push_back(c);
    g->stage_count[st] = static_cast<int>(list.size());
    if (!list.empty() && !pair)
      AKM_TRY(g->stage_list[st].upload(list.data(), int64_t(list.size())));
  }
  if (g->max_stages > 0 && !pair)
  {
    // first-stage groups: chains in order, grouped by (dimension, fill)
    std::vector<std::pair<int, int>> keys;
    std::vector<std::vector<int>> members;
    for (int c = 0; c < g->nchains; c++)
    {
      if (ch_nst[c] < 1)
        continue;
      const std::pair<int, int> key(ch_dim[c * gk_max_dims], ch_fill[c * gk_max_dims]);
      size_t i = 0;
      while (i < keys.size() && keys[i] != key)
        i++;
      if (i == keys.size())
      {
        keys.push_back(key);
        members.emplace_back();
      }
      members[i].push_back(c);
    }
    std::vector<int> gptr(1, 0), gchain;
    for (auto const &mem : members)
      for (size_t b = 0; b < mem.size(); b += gk_group_max)
      {
        for (size_t j = b; j < std::min(mem.size(), b + gk_group_max); j++)
          gchain.push_back(mem[j]);
        gptr.push_back(static_cast<int>(gchain.size()));
      }
    g->first_groups = static_cast<int>(gptr.size()) - 1;
    for (int i = 0; i < g->first_groups; i++)
      g->first_largest = std::max(g->first_largest, gptr[i + 1] - gptr[i]);
    AKM_TRY(g->first_ptr.upload(gptr.data(), int64_t(gptr.size())));
    AKM_TRY(g->first_chain.upload(gchain.data(), int64_t(gchain.size())));
  }
  g->fl_lanes = fibre_lanes(m, lists, term_act);
  // a pair handle plans slabs when it is to use or to time them
  if (!pair || g->fl_lanes > fl_lanes_default(g->max_stages))
    AKM_TRY(need_slabs(m, *g));
  if (!pair && nslots + g->ngroups > 0)
    AKM_TRY(g->work.allocate((int64_t(2) * nslots + g->ngroups) * g->cells * m.N *
                             int64_t(m.esize)));
  // flops as the reference counts them (src/asgard_kronmult_matrix.cpp:
  // 1389-1395): two per entry of the full DOF-level pattern of every
  // non-identity (term, dimension) on the padded set
  for (int t = 0; t < m.T; t++)
    for (int k = 0; k < d; k++)
      if (active_mask == nullptr || active_mask[t * d + k] != 0)
        g->flops += 2 * nnz_dim[k];
  m.gk = std::move(g);
  return pair ? AKM_SUCCESS : global_set_layout(m, default_layout(m, *m.gk));
}

int factored_build(akm_matrix_s &m, std::vector<int> const &elem)
{
  m.gk.reset();
  m.factored = false;
  if (m.T == 0 || m.rows == 0)
    return AKM_SUCCESS;
  std::vector<int> mask;
  bool finite = false;
  AKM_TRY(stored_factors(m, mask, finite));
  return finite ? factored_build_mask(m, elem, mask) : AKM_SUCCESS;
}

int factored_refresh(akm_matrix_s &m)
{
  if (m.T == 0 || m.rows == 0)
    return AKM_SUCCESS;
  // the tables of the present plans, wanted or not: one wait for both
  if (m.gk)
    AKM_TRY(global_tables(m));
  std::vector<int> mask;
  bool finite = false;
  AKM_TRY(stored_factors(m, mask, finite));
  if (!finite)
  {
    m.form_stamp += m.factored ? 1 : 0;
    m.factored = false;
    return AKM_SUCCESS;
  }
  // a factor that became the identity may stay in the products; one that was
  // the identity when the products were chosen may not change
  bool covered = m.gk != nullptr;
  for (size_t i = 0; covered && i < mask.size(); i++)
    covered = mask[i] <= m.factored_mask[i];
  if (covered)
  {
    m.form_stamp += m.factored ? 0 : 1;
    m.factored = true;
    return AKM_SUCCESS;
  }
  if (mask == m.factored_mask)
    return AKM_SUCCESS; // no factored form for these factors
  AKM_HIP(hipStreamSynchronize(m.stream));
  return factored_build_mask(m, m.elem_host, mask);
}

int factored_build_mask(akm_matrix_s &m, std::vector<int> const &elem, std::vector<int> const &mask)
{
  m.gk.reset();
  m.factored = false;
  m.factored_mask = mask;
  m.form_stamp++;
  m.pair_tuned = false; // it was timed against another form, or none
  int widest = 0;
  for (int t = 0; t < m.T; t++)
    widest = std::max(widest, static_cast<int>(std::count(mask.begin() + t * m.d,
                                                          mask.begin() + (t + 1) * m.d, 1)));
  // one non-identity dimension per term: a product along fibres, exact on
  // any cells; more: the chain split needs a standard grid
  if (widest > 1 && !whole_level_grid(m.d, m.rows, elem.data()))
    return AKM_SUCCESS;
  int64_t repeated = -1;
  int layout = -1;
  if (build_global(m, elem, mask.data(), nullptr, true, repeated) == AKM_SUCCESS && m.gk)
    layout = default_layout(m, *m.gk);
  // too large for the lists or for memory, or a cell repeated: the pair
  // kernels need neither
  if (layout < 0)
  {
    (void)hipGetLastError();
    m.gk.reset();
    return AKM_SUCCESS;
  }
  const akm_global_s &g = *m.gk;
  // Estimated times: the pair kernels' fixed part and rate, the fibre walk's
  // per launch and per step (the slab layout is taken where it is faster
  // than that).
  const double pair_us = 4.0 + double(m.flops()) / (m.prec == AKM_F64 ? 25e6 : 50e6);
  const double walk_us = 1.0 + 3.0 * std::max(g.max_stages, 1) + double(g.fl_lanes) / 0.6e6;
  m.factored = walk_us < pair_us && global_set_layout(m, layout) == AKM_SUCCESS;
  if (!m.factored)
  {
    (void)hipGetLastError();
    m.gk.reset();
  }
  return AKM_SUCCESS;
}
} // namespace akm

using namespace akm;

extern "C" {

akm_status akm_create_global_grid(int d, int n, int64_t num_cells, const int *table,
                                  int max_level, int T, const void *vA, int64_t num_vA,
                                  const int *active, const int *flux_dim, akm_prec prec,
                                  akm_matrix *mat)
{
  if (mat == nullptr)
    return set_error(AKM_ERR_INVALID, "null matrix handle pointer");
  *mat = nullptr;
  if (d < 1 || d > gk_max_dims)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: d = %d not in [1, 6]", d);
  if (n < 1 || n > 16)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: n = %d not in [1, 16]", n);
  if (num_cells < 0 || num_cells > (int64_t(1) << 31) - 2 || T < 0)
    return set_error(AKM_ERR_INVALID, "global kron: invalid sizes");
  if (prec != AKM_F64 && prec != AKM_F32)
    return set_error(AKM_ERR_INVALID, "global kron: unknown precision %d", int(prec));
  if (table == nullptr && num_cells > 0)
    return set_error(AKM_ERR_INVALID, "global kron: null table");
  if (max_level < 0 || max_level > 20)
    return set_error(AKM_ERR_INVALID, "global kron: max_level %d not in [0, 20]", max_level);
  for (int64_t c = 0; c < num_cells; c++)
    for (int k = 0; k < d; k++)
    {
      const int L = table[c * 2 * d + k], p = table[c * 2 * d + d + k];
      if (L < 0 || L > max_level || p < 0 || (L <= 1 && p != 0) ||
          (L > 1 && p >= (1 << (L - 1))))
        return set_error(AKM_ERR_INVALID, "global kron: invalid cell (%d, %d)", L, p);
    }
  std::vector<int> p1, i1, dg;
  AKM_TRY(build_connect_1d(max_level, true, p1, i1, dg));
  const int64_t nconn = static_cast<int64_t>(i1.size());
  const int64_t expect_vA = nconn * d * T * int64_t(n) * n;
  if (T > 0 && (vA == nullptr || num_vA != expect_vA))
    return set_error(AKM_ERR_INVALID,
                     "global kron: vA has %lld values, connect_1d(%d) needs %lld",
                     static_cast<long long>(num_vA), max_level,
                     static_cast<long long>(expect_vA));
  std::vector<int> elem;
  cell_1d_indices(d, num_cells, table, elem);
  std::unique_ptr<akm_matrix_s> m(new akm_matrix_s());
  m->prec = prec;
  m->esize = (prec == AKM_F64) ? 8 : 4;
  m->d = d;
  m->n = n;
  m->rows = m->cols = static_cast<int>(num_cells);
  m->T = T;
  int64_t N = 1;
  for (int k = 0; k < d; k++)
    N *= n;
  if (N > 4096)
    return set_error(AKM_ERR_UNSUPPORTED, "global kron: n^d = %lld exceeds 4096",
                     static_cast<long long>(N));
  m->N = N;
  m->mode = mode_global;
  m->max_level = max_level;
  m->M = 1 << max_level;
  m->num_vA = (T > 0) ? num_vA : 0;
  m->nconn = static_cast<int>(nconn);
  if (T > 0)
    AKM_TRY(m->vA.upload(static_cast<const unsigned char *>(vA), num_vA * m->esize));
  int64_t repeated = -1;
  AKM_TRY(build_global(*m, elem, active, flux_dim, false, repeated));
  if (repeated >= 0)
    return set_error(AKM_ERR_INVALID, "global kron: cell %lld repeated",
                     static_cast<long long>(repeated));
  if (T > 0)
    AKM_TRY(global_update(*m, vA));
  *mat = m.release();
  return AKM_SUCCESS;
}

akm_status akm_global_slab_info(akm_matrix mat, int *groups, int *rest_chains, int *sum_sources)
{
  if (mat == nullptr || mat->mode != mode_global || !mat->gk)
    return set_error(AKM_ERR_INVALID, "global slab info: not a global kron matrix");
  akm_global_s const &g = *mat->gk;
  if (groups)
    *groups = g.ngroups;
  if (rest_chains)
    *rest_chains = g.max_stages > 0 ? g.stage_count_rest[0] : 0;
  if (sum_sources)
    *sum_sources = g.nsrc_slab;
  return AKM_SUCCESS;
}

akm_status akm_global_info(akm_matrix mat, int64_t *padded_cells, int *chains, int *stages)
{
  if (mat == nullptr || mat->mode != mode_global || !mat->gk)
    return set_error(AKM_ERR_INVALID, "global info: not a global kron matrix");
  if (padded_cells)
    *padded_cells = mat->gk->cells - mat->gk->active_cells;
  if (chains)
    *chains = mat->gk->nchains;
  if (stages)
    *stages = mat->gk->max_stages;
  return AKM_SUCCESS;
}

akm_status akm_global_jacobi(akm_matrix mat, double *pc)
{
  if (mat == nullptr || mat->mode != mode_global || !mat->gk || pc == nullptr)
    return set_error(AKM_ERR_INVALID, "global jacobi: not a global kron matrix");
  const int64_t count = mat->gk->active_cells * mat->N;
  if (count > 0 && mat->gk->pc.data() != nullptr)
  {
    AKM_HIP(hipMemcpyAsync(pc, mat->gk->pc.data(), sizeof(double) * count, hipMemcpyDeviceToHost,
                           mat->stream));
    AKM_HIP(hipStreamSynchronize(mat->stream));
  }
  else if (count > 0)
    std::fill(pc, pc + count, 0.0);
  return AKM_SUCCESS;
}

} // extern "C"
