// Fibre lists of a cell set and the fibre-walk kernels built on them.
//
// A fibre along dimension k is a class of cells equal in every other 1D
// index.  A factor that acts in dimension k and is the identity elsewhere
// couples only cells of one fibre, so its product is a walk over the
// connect_1d row of a cell, restricted to the fibre's members.
#pragma once

#include <cstdint>
#include <vector>

#include "akm_internal.hpp"

struct akm_matrix_s;

namespace akm
{
//! Part of a 1D factor a product applies.
enum gk_fill : int
{
  gk_upper = 0, // from the diagonal on (diagonal included)
  gk_full = 1,
  gk_lower = 2, // strictly before the diagonal
};

//! Connected cells of every cell's fibre along one dimension, 1D index
//! ascending, with their connect_1d positions and the position of the cell
//! itself.
struct gk_lists
{
  std::vector<int> ptr, cell, q, diag;
};

//! Fibre lists along dimension k, and the cells fibre by fibre (fibres in
//! the order of their other 1D indices).  `repeated` = the first cell equal
//! to an earlier one, or -1.
int build_fibre_lists(int d, int64_t cells, const int *elem, int k, int M,
                      std::vector<int> const &c1_pntr, std::vector<int> const &c1_indx,
                      std::vector<int> const &c1_diag, gk_lists &out, std::vector<int> &order,
                      int64_t &repeated);

//! True when the cells are whole levels (every cell of each level vector
//! present) and the level vectors are closed under lowering any level: a
//! standard sparse or full grid.  The chain split of a product of 1D factors
//! is then exact for any factors.
bool whole_level_grid(int d, int64_t cells, const int *elem);

//! A launch-ready fibre-walk plan: the products of every term in dependent
//! stages.
struct fibre_plan
{
  struct stage
  {
    int first_group = 0, groups = 0; // workgroups in `slots`
  };
  bool built = false;
  bool slots_of_lanes = true; // fl_stage; else one workgroup per cell
  int tpb = 256, nslot = 1; // threads and slots per workgroup
  int vectors = 0;          // work vectors
  int identities = 0;       // terms of identity factors only
  std::vector<stage> stages;
  dev_buffer<int4> slots, pieces;
  dev_buffer<unsigned char> work, tab;
  // factor tables: table i sums the (term, dimension) pairs
  // tab_src[tab_ptr[i] .. tab_ptr[i+1]) of the vA the matrix had at `stamp`
  // (tab_def: tab_ptr, from src0 on tab_src, from diag0 on connect_1d's
  // diagonal positions)
  dev_buffer<int> tab_def;
  int src0 = 0, diag0 = 0;
  int ntab = 0, nconn = 0, M = 0;
  int64_t stride = 0; // work vector size
  bool tab_valid = false;
  uint64_t stamp = 0;
};

//! The products of all terms (term_act[t]: the term's non-identity
//! dimensions, the whole-acting one first) over the padded cells, as counted
//! by fibre_lanes and launched by fibre_apply.
int build_fibre_plan(akm_matrix_s const &m, int64_t active_cells, int64_t cells, const int *elem,
                     std::vector<gk_lists> const &lists,
                     std::vector<std::vector<int>> const &term_act,
                     std::vector<int> const &c1_diag, fibre_plan &plan);

//! A single-stage FP64 plan and its system's vectors (Krylov basis, solution,
//! size, time step) as the batch kernel reads them.
struct fibre_system
{
  const int4 *slots, *pieces;
  const double *tab;
  double *V, *X;
  int64_t size;
  double dt;
  int n, N, nslot, identities;
};
fibre_system fibre_batch_system(akm_matrix_s const &m, fibre_plan const &plan, double *V,
                                double *X, int64_t size, double dt);
//! Rebuilds the plan's factor tables on `stream` when vA changed.
int fibre_refresh(akm_matrix_s const &m, fibre_plan &plan, hipStream_t stream);
//! One workgroup of tpb threads per (system, group) of `items`.
int launch_fibre_batch(int tpb, int groups, const fibre_system *fs, const int2 *items,
                       const int *jcol, int joff, int limit, const int *active, int phase,
                       hipStream_t stream);
//! The plan of a sparse-grid FP64 matrix for a batch: true when its factored
//! form runs in one stage.
bool factored_batch_plan(akm_matrix_s const &m, fibre_plan &plan, int &rc);

//! (lane, connection) steps of one apply of the plan, without building it.
int64_t fibre_lanes(akm_matrix_s const &m, std::vector<gk_lists> const &lists,
                    std::vector<std::vector<int>> const &term_act);

//! y = (alpha*A*x + beta*y + gamma*xg) / (1 - jdt*pc) (no division when pc is
//! null).
template<typename P>
int fibre_apply(akm_matrix_s &m, fibre_plan &plan, P alpha, const P *x, P beta, P *y, P gamma,
                const P *xg, const double *pc, double jdt);

//! w = v + c * fp64(A fp32(v)) of an FP32 operator on FP64 vectors, in one
//! launch; false when the plan has several stages.
bool fibre_apply_between(akm_matrix_s &m, fibre_plan &plan, const double *v, double c, double *w);
} // namespace akm
