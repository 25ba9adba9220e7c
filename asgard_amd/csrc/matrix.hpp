// The kronmult matrix object behind the akm_matrix handle.
#pragma once

#include <memory>
#include <mutex>
#include <vector>

#include "akm_internal.hpp"
#include "kron_kernels.hpp"

struct akm_gmres_workspace;
struct akm_global_s;

struct akm_matrix_s
{
  akm_prec prec = AKM_F64;
  int d = 0, n = 0, rows = 0, cols = 0, T = 0;
  int mode = akm::mode_ia;
  int64_t N = 1;   // tensor size n^d
  int64_t nnz = 0; // connected (row, col) pairs
  size_t esize = 8;

  // sparse: CSR (host row pointer kept for work decomposition)
  std::vector<int64_t> pntr;
  akm::dev_buffer<int> indx, iA;
  akm::dev_buffer<unsigned char> vA;
  int64_t num_vA = 0;
  // advanced by every call that rewrites vA, so that a batch knows when to
  // rebuild the tables of its plans
  uint64_t vA_stamp = 0;
  // the first implicit solve's timed operator apply (ms; -1 before it),
  // which decides whether GMRES steps are enqueued ahead
  double gmres_apply_ms = -1;
  // grid mode
  akm::dev_buffer<int> elem, off1d;
  int M = 0;
  int max_level = 0;
  // grid mode, LDS factor tables: factors as [dim][connection][term][nnp],
  // connect_1d row pointer, packed cell 1D indices
  akm::dev_buffer<unsigned char> vAk;
  akm::dev_buffer<int> conn_pntr;
  akm::dev_buffer<unsigned long long> epack;
  std::vector<int> conn_pntr_host, conn_indx_host, conn_diag_host;
  int nconn = 0, nnp = 0;
  int64_t max_table_elems = 0;
  int64_t max_table_last4 = 0; // largest per-row table of the last four dimensions
  int lds_cap = -1; // -1 automatic, 0 disables the LDS tables
  // dense mode
  std::vector<akm::dev_buffer<unsigned char>> terms;
  akm::dev_buffer<void *> term_ptrs;
  int nb = 0, row_offset = 0, col_offset = 0;

  // work decomposition: one workgroup per row, rows longest first
  int waves = 0;        // wavefronts per row workgroup (0 = automatic)
  int force_generic = 0;
  int family = 0;       // 0 register / LDS-table kernels, 1 matrix-core kernel
  akm::dev_buffer<int64_t> pntr_dev;
  akm::dev_buffer<int> row_order;

  // workspaces for host-resident vectors
  akm::dev_buffer<unsigned char> xws, yws;

  // operator update on the device: connect_1d (rows, then columns) in vA
  // order and the scan's findings, and the device copy of the caller's operator pointers
  akm::dev_buffer<int> op_conn;
  int op_scan = 0; // number of the last scan of the stored factors
  akm::dev_buffer<const void *> op_ptrs;
  // IMEX step vectors (four of output_size), on the implicit handle
  akm::dev_buffer<double> imex_ws;

  hipStream_t stream = nullptr;

  std::unique_ptr<akm_gmres_workspace, void (*)(akm_gmres_workspace *)> gmres{nullptr,
                                                                             nullptr};
  // sparse-grid handles: the operator runs one dimension at a time (gk)
  // instead of pair by pair, because its factors allow it
  bool factored = false;
  // advanced when the form or the products it was built for change
  uint64_t form_stamp = 0;
  bool pair_kernels = false;        // the caller asked for the pair kernels
  bool pair_tuned = false;          // akm_autotune found them faster than the form
  // held while a factored apply is enqueued: its launches share work vectors,
  // so two threads' applies follow each other on the stream
  std::mutex factored_mtx;
  std::vector<int> factored_mask;   // T x d non-identity factors gk was built for
  std::vector<int> elem_host;       // cell 1D indices
  // global Kronecker operator (mode_global), or the factored form of a
  // sparse-grid operator
  std::unique_ptr<akm_global_s, void (*)(akm_global_s *)> gk{nullptr, nullptr};

  int64_t input_size() const { return N * cols; }
  int64_t output_size() const { return N * rows; }
  int64_t flops() const;
};

namespace akm
{
//! y = alpha*A*x + beta*y + gamma*xg on device pointers (xg row-indexed).
int apply_device(akm_matrix_s &m, double alpha, const void *x, double beta, void *y,
                 double gamma, const void *xg);

//! Moves the handle to `stream`.  Where applies share work vectors of the
//! handle, the new stream waits for what still runs on the old one (unless
//! either is being captured).
void use_stream(akm_matrix_s &m, hipStream_t stream);

//! Wavefronts per row workgroup used for the matrix (explicit or automatic).
int waves_per_row(akm_matrix_s const &m);

//! Global operator: y = alpha*A*x + beta*y + gamma*xg on device pointers,
//! divided by (1 - jdt * pc) with the reference's Jacobi diagonal when
//! `jacobi` is set.
int global_apply(akm_matrix_s &m, double alpha, const void *x, double beta, void *y,
                 double gamma, const void *xg, bool jacobi, double jdt);
//! w = v + c * fp64(A fp32(v)) of an FP32 operator in one launch on FP64
//! vectors, when its form has one (a fibre walk of one stage); false, with
//! nothing enqueued, otherwise.
bool apply_f32_between(akm_matrix_s &m, const double *v, double c, double *w);
//! Global operator: new factor values (same vA layout), Jacobi diagonal rebuilt.
int global_update(akm_matrix_s &m, const void *vA);
//! Global operator: Jacobi diagonal rebuilt on the device from the stored
//! factor blocks (after they were written on the device).
int global_device_jacobi(akm_matrix_s &m);
//! Rebuilds the factor tables of every plan the handle has from the stored
//! factors, in place.  An apply never does: it may be captured into a graph,
//! or be the first after one was.
int global_tables(akm_matrix_s &m);
//! Fills vAk from vA: the factors re-laid from [connection][term][dim][n*n] to
//! [dim][connection][term][nnp] for the LDS-table kernel, so that the blocks
//! one row's 1D cell can touch in one dimension are one contiguous range.
int relayout_factors(akm_matrix_s &m);

//! Which of a sparse-grid handle's T x d stored factors are not exactly the
//! identity, and whether all their values are finite: scanned on the device.
int stored_factors(akm_matrix_s &m, std::vector<int> &mask, bool &finite);
//! Sparse-grid handle: builds the factored form of its operator (`elem`: cell
//! 1D indices) when the stored factors allow one that is faster than the pair
//! kernels.
int factored_build(akm_matrix_s &m, std::vector<int> const &elem);
//! After new factor values: keeps the factored form when it still holds, else
//! builds it anew.
int factored_refresh(akm_matrix_s &m);
//! The same as factored_build for known non-identity factors (mask, T x d, all values finite).
int factored_build_mask(akm_matrix_s &m, std::vector<int> const &elem,
                        std::vector<int> const &mask);
//! Global operator: flops per apply as the reference counts them.
int64_t global_flops(akm_matrix_s const &m);
//! Global operator: row layout in use, as akm_set_tuning takes it (1, 8, 2,
//! 3, 4, 5 or 6).
int global_layout(akm_matrix_s const &m);
//! Dependent products of its longest chain.
int global_stages(akm_matrix_s const &m);
//! True when its applies write work vectors of the handle, so that two of them
//! must not run at once.
bool global_shares_work(akm_matrix_s const &m);
//! Global operator: times the layouts on the operator and keeps the fastest;
//! best_ms = its time per apply.
int global_autotune(akm_matrix_s &m, const void *x, void *y, double &best_ms);
//! Factored sparse-grid operator: the layout and stream split in use, as one
//! number, and back.
int factored_shape(akm_matrix_s const &m);
int factored_set_shape(akm_matrix_s &m, int shape);
//! Global operator: row layout 1 (lane per DOF), 8 (the fibre walk, lists
//! split over slots of lanes), 2 (wavefront per cell), 3 (wavefront per cell, chains sharing their first
//! stage's input read it once), 4 / 5 (2 / 3 with each XCD taking contiguous
//! cells), 6 (slabs), 0 (unchanged).
int global_set_layout(akm_matrix_s &m, int layout);

//! Kernel arguments of an FP64 matrix (vectors and scalars left empty).
kron_args<double> kron_args_f64(akm_matrix_s const &m);
} // namespace akm
