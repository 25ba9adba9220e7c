// Sparse-grid index construction (1D hierarchy connectivity, cell 1D indices
// and the GPU cell-pair pattern scan).
#pragma once

#include <cstdint>
#include <vector>

#include "akm_internal.hpp"

namespace akm
{
//! connect_1d: CSR over the 2^max_level 1D cells, columns ascending.
int build_connect_1d(int max_level, bool full, std::vector<int> &pntr, std::vector<int> &indx,
                     std::vector<int> &diag);

//! Dense M x M table (M = 2^max_level) of connect_1d positions, -1 when the
//! two 1D cells are not connected; pntr and indx are connect_1d(max_level).
int build_offset_table(int max_level, std::vector<int> const &pntr, std::vector<int> const &indx,
                       std::vector<int> &table);

//! The indices 0 .. keys.size()-1 ordered by key (the lowest `bits` bits hold
//! it), equal keys by index, by radix passes (handles are built at every
//! regrid; 16,172 cells in 42 bits 0.12 ms with the keys, a comparison sort 0.6).
void radix_order(std::vector<uint64_t> const &keys, int bits, std::vector<int> &order);

//! elem[c*d + k] = 1D index of cell c in dimension k (0 for level 0, else
//! 2^(level-1) + position).
void cell_1d_indices(int d, int64_t num_cells, const int *table, std::vector<int> &elem);

//! Cell-pair CSR on the GPU: pntr (host) and the column ids (device), each
//! row's columns ascending, or in the order of order_host (a permutation of
//! the cells) when it is not null.
int device_sparse_pattern(int d, int64_t num_cells, const int *table_host,
                          std::vector<int64_t> &pntr, dev_buffer<int> &indx_dev,
                          const int *order_host = nullptr);

//! The same for valid cells below level 11, given by their packed 1D indices
//! (10 bits a dimension) and connect_1d(max_level); each row's columns in the
//! order of order_host, a permutation of the cells.  The row starts stay on
//! the device, too.
int device_sparse_pattern(int d, std::vector<uint64_t> const &pack, int max_level,
                          std::vector<int> const &c1_pntr, std::vector<int> const &c1_indx,
                          std::vector<int> const &order_host, std::vector<int64_t> &pntr,
                          dev_buffer<int64_t> &pntr_dev, dev_buffer<int> &indx_dev);

//! The cells 0 .. cells-1 ordered by their 1D indices in `dims` (the first
//! the most significant), ties by cell id; 1D indices are below M.
void order_by_dims(int d, int64_t cells, const int *elem, std::vector<int> const &dims, int M,
                   std::vector<int> &order);

//! The cells sorted lexicographically by their 1D indices (dimension 0
//! first), ties by cell id.
void lexicographic_order(int d, int64_t num_cells, const int *elem, std::vector<int> &order);
} // namespace akm
