// Fibre-walk kernels: operators whose factors are mostly the identity, one
// dimension at a time, with no intermediate list of cell pairs.
//
// A term with non-identity dimensions S (a_0 the whole-acting one, then a_1
// .. a_{m-1}) is evaluated by the recursion
//   Op_0 = F_{a0},   Op_i v = L_{ai} (Op_{i-1} v) + Op_{i-1} (U_{ai} v)
// (F the whole factor, U its part from the diagonal on, L the part strictly
// before it), which is the sum of the 2^(m-1) chains of the reference's
// global operator (kronmult::permutes, src/device/asgard_kronmult.hpp:152-220)
// with the products that chains share taken once: 3 * 2^(m-1) - 2 products
// instead of m * 2^(m-1).  Products whose inputs are ready run in one launch,
// so a term takes m launches, and terms that act in one and the same single
// dimension are added into one factor table.
//
// Kernel: a workgroup holds `nslot` slots of N = n^d lanes.  A slot walks
// pieces of one cell's connection list, up to fl_piece connections each; a
// cell with a long list takes several slots of one workgroup, whose partials
// are added in slot order through LDS.  Lane e reads entry e of a connected
// cell's tensor once and multiplies it with its digit's column of the factor
// block, which gives it a share of the n rows of its fibre; the rows are
// summed through LDS at the end (reading row entries instead costs n loads of
// x per connection).  Results repeat bit for bit.
//
// What bounds it: on the operators it is chosen for, the chain of dependent
// loads and the launch, not bandwidth.  A piece's list entries sit in the
// slot's record, so the chain is record, blocks, LDS, store; lists are cut
// into pieces so that a row of 512 connections (a level-0 cell at d = 4,
// level 7) is not the tail of the launch.  Measured (FP64, us per apply, the
// pair kernels and the best other global layout before): d = 4 n = 2 level 7
// advection-diffusion 7.1 (411 / 20); d = 4 n = 3 level 5 9.5 (129 / 12);
// d = 2 n = 2 level 5 3.3 (3.9 / 6.5); d = 3 n = 3 level 6, every factor
// dense, three stages 24 (23 / 60).
#include "fibre.hpp"
#include "grid.hpp"
#include "kron_kernels.hpp"
#include "matrix.hpp"

#include <algorithm>
#include <array>
#include <deque>
#include <map>
#include <memory>
#include <type_traits>

namespace akm
{
namespace
{
constexpr int fl_piece = 8; // connections of a piece: one batch of loads

//! Up to fl_piece connections of one product.
struct fl_piece_rec
{
  int in;     // vector: 0 the operator's input, v > 0 work vector v - 1
  int stride; // tensor stride of the product's dimension
  unsigned magic; // ceil(2^32 / stride), 0 for stride 1
  int len;        // connections | last piece of its round << 16
  // (connected cell, factor block of all tables); entries past len name the
  // zero block
  int2 entry[fl_piece];
};
static_assert(sizeof(fl_piece_rec) == 5 * sizeof(int4), "piece records are five int4");

//! A slot and its first piece.
struct fl_slot_rec
{
  int cell;  // output cell, -1: empty slot
  int group; // rank within the cell's slots | slots << 16
  int vec;   // output work vector, -1: y
  int more;  // further pieces: more of them from `next` on
  int next, rounds, pad[2]; // rounds: of the workgroup (the same in its slots)
  fl_piece_rec p;
};
static_assert(sizeof(fl_slot_rec) == 7 * sizeof(int4), "slot records are seven int4");

//! P: values of the factors, work vectors and sums; X: of the input and y.
template<typename P, typename X = P>
struct fl_args
{
  const int4 *slots;
  const int4 *pieces;
  const P *tab;
  int n, N, nslot;
  int64_t stride;
  const X *x;
  P *work;
  X *y;
  const X *xg;
  const double *pc;
  double jdt;
  P alpha, beta, gamma;
  double between; // X != P: y = xg + between * sum
  int identities;
};

//! Column s of a factor block, n values.
template<typename P, int NT>
__device__ __forceinline__ void fl_column(const P *A, P (&v)[NT])
{
  constexpr int W = (NT % 2 != 0) ? 1 : ((sizeof(P) == 4) ? NT : 2); // values per read
  typedef P vec __attribute__((ext_vector_type(W)));
#pragma unroll
  for (int j = 0; j < NT; j += W)
  {
    const vec t = *reinterpret_cast<const vec *>(A + j);
#pragma unroll
    for (int i = 0; i < W; i++)
      v[j + i] = t[i];
  }
}

//! Digit of tensor entry e at the piece's dimension.
__device__ __forceinline__ int fl_digit(int e, unsigned magic, int n)
{
  return ((magic != 0) ? static_cast<int>(__umulhi(static_cast<unsigned>(e), magic)) : e) % n;
}

//! c[r] += the first U of a piece's connections: column `s` of each block
//! times entry e of the connected cell.  All loads precede their uses.
template<typename P, typename X, int NT, int U>
__device__ __forceinline__ void fl_connections(const X *__restrict__ in, const P *__restrict__ tab,
                                               int N, int len, const int4 *ent, P (&c)[NT])
{
  P av[U][NT], xv[U];
#pragma unroll
  for (int u = 0; u < U; u++)
  {
    const int cell = (u % 2 == 0) ? ent[u / 2].x : ent[u / 2].z;
    const int block = (u % 2 == 0) ? ent[u / 2].y : ent[u / 2].w;
    xv[u] = static_cast<P>(in[int64_t(cell) * N]);
    fl_column<P, NT>(tab + int64_t(block) * (NT * NT), av[u]);
  }
#pragma unroll
  for (int u = 0; u < U; u++)
  {
    const P xu = (u < len) ? xv[u] : P{0};
#pragma unroll
    for (int r = 0; r < NT; r++)
      c[r] = fma(av[u][r], xu, c[r]);
  }
}

//! A finished sum of entry pos of a vector: into its work vector, or into y.
template<typename P, typename X>
__device__ __forceinline__ void fl_store(fl_args<P, X> const &a, int vec, int64_t pos, P sum)
{
  if constexpr (!std::is_same_v<P, X>)
  {
    if (a.identities > 0)
      sum += static_cast<P>(a.identities) * static_cast<P>(a.x[pos]);
    a.y[pos] = fma(a.between, static_cast<X>(sum), a.xg[pos]);
    return;
  }
  if (vec >= 0)
  {
    a.work[int64_t(vec) * a.stride + pos] = sum;
    return;
  }
  if (a.identities > 0)
    sum += static_cast<P>(a.identities) * a.x[pos];
  P out = a.alpha * sum;
  if (a.beta != P{0})
    out += a.beta * a.y[pos];
  if (a.gamma != P{0})
    out += a.gamma * a.xg[pos];
  if (a.pc != nullptr)
    out = static_cast<P>(static_cast<double>(out) / (1.0 - a.jdt * a.pc[pos]));
  a.y[pos] = out;
}

//! One workgroup's slots, then each cell's slot partials added in slot order.
//! A slot whose pieces act in several dimensions takes a round per dimension.
//! LDS: NT values per thread.
template<typename P, int NT, typename X>
__device__ __forceinline__ void fl_group(fl_args<P, X> const &a, int64_t group, P *ex)
{
  const int tpb = blockDim.x, t = threadIdx.x, N = a.N;
  const int slot = t / N;
  const int e = t - slot * N;
  const bool mine = slot < a.nslot;
  // idle lanes read slot 0's record and store nothing
  const int4 *rec = a.slots + (group * a.nslot + (mine ? slot : 0)) * 7;
  const int4 head = rec[0], tail = rec[1];
  int4 ph = rec[2];
  int4 ent[fl_piece / 2] = {rec[3], rec[4], rec[5], rec[6]};
  const bool live = mine && head.x >= 0;
  int more = live ? head.w : 0;
  const int4 *next = a.pieces + int64_t(tail.x) * 5;
  bool have = live;
  P acc = 0;
  const int rounds = tail.y;
  for (int round = 0; round < rounds; round++)
  {
    P c[NT];
#pragma unroll
    for (int r = 0; r < NT; r++)
      c[r] = 0;
    const int s = fl_digit(e, static_cast<unsigned>(ph.z), NT);
    const int stride = ph.y;
    bool open = have;
    while (open)
    {
      const int len = ph.w & 0xffff;
      open = (ph.w >> 16) == 0;
      const X *in = a.x + e;
      if constexpr (std::is_same_v<P, X>)
        in = ((ph.x == 0) ? a.x : a.work + int64_t(ph.x - 1) * a.stride) + e;
      const int4 cur[fl_piece / 2] = {ent[0], ent[1], ent[2], ent[3]};
      have = more > 0;
      if (have)
      {
        ph = next[0];
#pragma unroll
        for (int i = 0; i < fl_piece / 2; i++)
          ent[i] = next[1 + i];
        next += 5;
        more--;
      }
      const P *tab = a.tab + s * NT;
      if (NT == 4)
      {
        // eight blocks' columns of four values do not fit the registers
        fl_connections<P, X, NT, fl_piece / 2>(in, tab, N, len, cur, c);
        if (__any(len > fl_piece / 2))
          fl_connections<P, X, NT, fl_piece / 2>(in, tab, N, len - fl_piece / 2,
                                                 cur + fl_piece / 4, c);
      }
      else if (__any(len > fl_piece / 2))
        fl_connections<P, X, NT, fl_piece>(in, tab, N, len, cur, c);
      else
        fl_connections<P, X, NT, fl_piece / 2>(in, tab, N, len, cur, c);
    }
    // lane e holds shares of the rows of its fibre: row r's entry is e with
    // its digit s replaced by r
    if (mine)
    {
#pragma unroll
      for (int r = 0; r < NT; r++)
        ex[s * tpb + t + (r - s) * stride] = c[r];
    }
    __syncthreads();
    if (round + 1 == rounds)
      break;
#pragma unroll
    for (int r = 0; r < NT; r++)
      acc += ex[r * tpb + t];
    __syncthreads();
  }
  if (rounds > 1)
  {
    // earlier rounds' sums join the last round's shares
    const P last = ex[t];
    __syncthreads();
    ex[t] = acc + last;
    __syncthreads();
  }
  if (!live || (head.y & 0xffff) != 0)
    return;
  P sum = 0;
  const int count = head.y >> 16;
  for (int i = 0; i < count; i++)
  {
#pragma unroll
    for (int r = 0; r < NT; r++)
      sum += ex[r * tpb + t + i * N];
  }
  fl_store(a, head.z, int64_t(head.x) * N + e, sum);
}

//! One stage: a workgroup per group of slots from group0 on.
template<typename P, int NT, int TPB, typename X>
__global__ void __launch_bounds__(TPB) fl_stage(fl_args<P, X> a, int group0)
{
  extern __shared__ __align__(16) unsigned char fl_smem[];
  fl_group<P, NT, X>(a, group0 + blockIdx.x, reinterpret_cast<P *>(fl_smem));
}

//! The single stage of every system of a batch: workgroup b takes group
//! items[b].y of system items[b].x.  Phase 0 forms the residual of every active
//! system, V[0] = b - (I - dt A) x (V[0] holds b on entry); phase 1 applies
//! the implicit operator to Krylov column j = *jcol + joff < limit, V[j+1] =
//! (I - dt A) V[j].
//! Workgroups of 1024 threads serve tensors of 65 entries on, which in a
//! batch have n = 3.
template<int TPB>
__global__ void __launch_bounds__(TPB)
    fl_batch(const fibre_system *__restrict__ fs, const int2 *__restrict__ items,
             const int *jcol, int joff, int limit, const int *active, int phase)
{
  extern __shared__ __align__(16) unsigned char fl_smem[];
  double *ex = reinterpret_cast<double *>(fl_smem);
  const int2 item = items[blockIdx.x];
  // the same in every lane: the system's record is read by scalar loads
  const int s = __builtin_amdgcn_readfirstlane(item.x);
  const int j = *jcol + joff;
  const fibre_system f = fs[s];
  if (active[s] == 0 || (phase != 0 && j >= limit))
    return;
  fl_args<double> a{};
  a.slots = f.slots;
  a.pieces = f.pieces;
  a.tab = f.tab;
  a.N = f.N;
  a.nslot = f.nslot;
  a.identities = f.identities;
  a.x = (phase == 0) ? f.X : f.V + int64_t(j) * f.size;
  a.y = (phase == 0) ? f.V : f.V + int64_t(j + 1) * f.size;
  a.xg = a.x;
  a.alpha = (phase == 0) ? f.dt : -f.dt;
  a.beta = (phase == 0) ? 1.0 : 0.0;
  a.gamma = (phase == 0) ? -1.0 : 1.0;
  const int64_t group = __builtin_amdgcn_readfirstlane(item.y);
  if (TPB == 1024 || f.n == 3)
    fl_group<double, 3, double>(a, group, ex);
  else if (f.n == 2)
    fl_group<double, 2, double>(a, group, ex);
  else
    fl_group<double, 4, double>(a, group, ex);
}

//! One stage for n > 4 or N > 1024: a workgroup per job and up to fl_any_width
//! of the cell's entries, row by row.  Its threads form groups of that many,
//! which take the pieces of the cell's list in turn (one group alone walked
//! the 256 connections of a level-0 cell at d = 2, n = 5, level 7 for 136 us)
//! and whose sums meet in LDS in group order.  NT: n where it is known, else 0.
//! Measured (FP64, us per apply; one group / groups / pair kernels / best other
//! global layout): d = 2 n = 5 level 7 136 / 12 / 23 / 51; d = 3 n = 5 level 6
//! 109 / 30 / 175 / 59; d = 2 n = 6 level 6 80 / 20 / 1352 / 56; d = 4 n = 6
//! level 3 132 / 16 / 3984 / 19.
constexpr int fl_any_width = 256;
template<typename P, int NT, int TPB>
__global__ void __launch_bounds__(TPB) fl_stage_any(fl_args<P> a, int group0)
{
  __shared__ P part[TPB];
  const int4 *rec = a.slots + int64_t(group0 + blockIdx.x) * 7;
  const int4 head = rec[0], tail = rec[1];
  const int n = (NT > 0) ? NT : a.n;
  const int width = min(a.N, fl_any_width), groups = TPB / width;
  const int g = threadIdx.x / width, lane = threadIdx.x - g * width;
  const int e = blockIdx.y * fl_any_width + lane;
  P sum = 0;
  if (g < groups && e < a.N)
  {
    for (int i = g; i <= head.w; i += groups)
    {
      const int4 *p = (i == 0) ? rec + 2 : a.pieces + int64_t(tail.x + i - 1) * 5;
      const int4 ph = p[0];
      const int s = fl_digit(e, static_cast<unsigned>(ph.z), n);
      const P *in = ((ph.x == 0) ? a.x : a.work + int64_t(ph.x - 1) * a.stride) + e - s * ph.y;
      const int2 *ent = reinterpret_cast<const int2 *>(p + 1);
      const int len = ph.w & 0xffff;
#pragma unroll 4
      for (int u = 0; u < len; u++)
      {
        const P *A = a.tab + int64_t(ent[u].y) * (int64_t(n) * n) + s;
        const P *xin = in + int64_t(ent[u].x) * a.N;
#pragma unroll
        for (int j = 0; j < n; j++)
          sum = fma(A[j * n], xin[j * ph.y], sum);
      }
    }
  }
  part[threadIdx.x] = sum;
  __syncthreads();
  if (g != 0 || e >= a.N)
    return;
  for (int i = 1; i < min(groups, head.w + 1); i++)
    sum += part[i * width + lane];
  fl_store(a, head.z, int64_t(head.x) * a.N + e, sum);
}

//! Factor tables: block q of table i is the sum over its (term, dimension)
//! pairs of connect_1d block q (column-major, as in vA); then per 1D cell the
//! diagonal blocks cut to the columns from the row's own on (upper) and
//! before it (lower).  The last block of all is zero.
template<typename P>
__global__ void __launch_bounds__(256)
    fl_tables(const P *__restrict__ vA, const int *__restrict__ ptr, const int *__restrict__ src,
              const int *__restrict__ c1_diag, int ntab, int nconn, int M, int n, int d, int T,
              P *tab)
{
  const int nn = n * n;
  const int64_t per = int64_t(nconn + 2 * M) * nn;
  for (int64_t i = blockIdx.x * int64_t(256) + threadIdx.x; i < per * ntab + nn;
       i += int64_t(256) * gridDim.x)
  {
    const int t = static_cast<int>(i / per);
    const int64_t rem = i - t * per;
    const int b = static_cast<int>(rem / nn);
    const int w = static_cast<int>(rem - int64_t(b) * nn);
    const int j = w / n, s = w - j * n;
    int q = b;
    bool keep = t < ntab;
    if (keep && b >= nconn)
    {
      const bool upper = b < nconn + M;
      q = c1_diag[b - nconn - (upper ? 0 : M)];
      keep = upper ? j >= s : j < s;
    }
    P v = 0;
    if (keep)
      for (int k = ptr[t]; k < ptr[t + 1]; k++)
        v += vA[((int64_t(q) * T + src[2 * k]) * d + src[2 * k + 1]) * nn + w];
    tab[i] = v;
  }
}

//! One product of the plan before it is laid out.
struct product
{
  int in, out; // vectors: 0 the input, v > 0 work vector v - 1; out -1: y
  int k, fill, table, stage;
};

//! The products of all terms, in stages (see the file comment).
struct program
{
  std::vector<product> prods;
  std::vector<std::vector<std::pair<int, int>>> tables; // (term, dimension) pairs
  int vectors = 0, stages = 0, identities = 0;

  program(int T, std::vector<std::vector<int>> const &term_act)
  {
    std::map<int, int> single; // dimension -> table of the one-dimension terms
    for (int t = 0; t < T; t++)
    {
      act = term_act[t];
      const int m = static_cast<int>(act.size());
      if (m == 0)
      {
        identities++;
        continue;
      }
      stages = std::max(stages, m);
      table_of.assign(m, -1);
      if (m == 1)
      {
        auto it = single.find(act[0]);
        if (it != single.end())
        {
          tables[it->second].emplace_back(t, act[0]);
          continue;
        }
        single.emplace(act[0], static_cast<int>(tables.size()));
      }
      for (int i = 0; i < m; i++)
      {
        table_of[i] = static_cast<int>(tables.size());
        tables.push_back({{t, act[i]}});
      }
      upper.clear();
      partial.clear();
      emit(m - 1, 0, -1, m - 1);
    }
    // a product's stage is where its output is formed; y is formed last
    for (auto &p : prods)
      if (p.out < 0)
        p.stage = std::max(stages, 1) - 1;
  }

private:
  std::vector<int> act, table_of;
  std::map<int, int> upper;                    // set of uppers -> vector
  std::map<std::pair<int, int>, int> partial;  // (i, set) -> vector Op_i u_set

  //! u_set: the uppers of `set` (bits over act), the highest first.
  int upper_vector(int set)
  {
    if (set == 0)
      return 0;
    auto it = upper.find(set);
    if (it != upper.end())
      return it->second;
    int low = 0; // the lowest bit acts last
    while (((set >> low) & 1) == 0)
      low++;
    const int rest = set & (set - 1);
    const int in = upper_vector(rest);
    const int v = ++vectors;
    prods.push_back({in, v, act[low], gk_upper, table_of[low], __builtin_popcount(rest)});
    upper.emplace(set, v);
    return v;
  }
  //! Adds Op_i u_set to vector `out`, formed in stage `stage`.
  void emit(int i, int set, int out, int stage)
  {
    if (i == 0)
    {
      prods.push_back({upper_vector(set), out, act[0], gk_full, table_of[0], stage});
      return;
    }
    const std::pair<int, int> key(i - 1, set);
    auto it = partial.find(key);
    if (it == partial.end())
    {
      const int v = ++vectors;
      it = partial.emplace(key, v).first;
      emit(i - 1, set, v, __builtin_popcount(set) + i - 1);
    }
    prods.push_back({it->second, out, act[i], gk_lower, table_of[i], stage});
    emit(i - 1, set | (1 << i), out, stage);
  }
};

//! The part [lo, hi) of a cell's list a fill walks.
static void fill_range(gk_lists const &l, int cell, int fill, int &lo, int &hi)
{
  lo = (fill == gk_upper) ? l.diag[cell] : l.ptr[cell];
  hi = (fill == gk_lower) ? l.diag[cell] + 1 : l.ptr[cell + 1];
}
} // namespace

int build_fibre_lists(int d, int64_t cells, const int *elem, int k, int M,
                      std::vector<int> const &c1_pntr, std::vector<int> const &c1_indx,
                      std::vector<int> const &c1_diag, gk_lists &out, std::vector<int> &order,
                      int64_t &repeated)
{
  std::vector<int> dims;
  for (int j = 0; j < d; j++)
    if (j != k)
      dims.push_back(j);
  dims.push_back(k);
  order_by_dims(d, cells, elem, dims, M, order);
  repeated = -1;
  // fibre by fibre: every member's connections one after another, then each
  // cell's piece to its place
  struct link
  {
    int cell, q;
  };
  std::vector<int> member(M, -1), first(cells);
  std::vector<link> found;
  found.reserve(size_t(cells) * 4);
  out.ptr.assign(cells + 1, 0);
  out.diag.assign(cells, -1);
  for (int64_t f0 = 0; f0 < cells;)
  {
    const int *lead = elem + int64_t(order[f0]) * d;
    int64_t f1 = f0;
    for (; f1 < cells; f1++)
    {
      const int *cell = elem + int64_t(order[f1]) * d;
      bool same = true;
      for (int j = 0; j < d && same; j++)
        same = (j == k) || cell[j] == lead[j];
      if (!same)
        break;
      if (member[cell[k]] >= 0 && (repeated < 0 || order[f1] < repeated))
        repeated = order[f1];
      member[cell[k]] = order[f1];
    }
    const int last = elem[int64_t(order[f1 - 1]) * d + k];
    for (int64_t f = f0; f < f1; f++)
    {
      const int c = order[f], r = elem[int64_t(c) * d + k];
      const size_t begin = found.size();
      for (int q = c1_pntr[r]; q < c1_pntr[r + 1]; q++)
      {
        const int col = c1_indx[q];
        if (col > last)
          break;
        if (member[col] < 0)
          continue;
        if (q == c1_diag[r])
          out.diag[c] = static_cast<int>(found.size() - begin);
        found.push_back(link{member[col], q});
      }
      if (found.size() > (size_t(1) << 31) - 1)
        return set_error(AKM_ERR_UNSUPPORTED, "global kron: connection lists too large");
      first[c] = static_cast<int>(begin);
      out.ptr[c + 1] = static_cast<int>(found.size() - begin);
    }
    for (int64_t f = f0; f < f1; f++)
      member[elem[int64_t(order[f]) * d + k]] = -1;
    f0 = f1;
  }
  if (repeated >= 0)
    return AKM_SUCCESS;
  for (int64_t c = 0; c < cells; c++)
    out.ptr[c + 1] += out.ptr[c];
  out.cell.resize(found.size());
  out.q.resize(found.size());
  for (int64_t c = 0; c < cells; c++)
  {
    const int base = out.ptr[c];
    if (out.diag[c] >= 0)
      out.diag[c] += base;
    for (int i = 0; i < out.ptr[c + 1] - base; i++)
    {
      out.cell[base + i] = found[first[c] + i].cell;
      out.q[base + i] = found[first[c] + i].q;
    }
  }
  for (int64_t c = 0; c < cells; c++)
    if (out.diag[c] < 0 || out.cell[out.diag[c]] != c)
      return set_error(AKM_ERR_INVALID, "global kron: connect_1d row without its diagonal");
  return AKM_SUCCESS;
}

bool whole_level_grid(int d, int64_t cells, const int *elem)
{
  std::map<std::array<signed char, 6>, int64_t> levels;
  std::array<signed char, 6> key{}, last{};
  int64_t *last_count = nullptr;
  for (int64_t c = 0; c < cells; c++)
  {
    for (int k = 0; k < d; k++)
    {
      const int e = elem[c * d + k];
      key[k] = (e == 0) ? 0 : static_cast<signed char>(32 - __builtin_clz(unsigned(e)));
    }
    if (last_count == nullptr || key != last)
    {
      last_count = &levels[key];
      last = key;
    }
    ++*last_count;
  }
  for (auto const &kv : levels)
  {
    int64_t whole = 1;
    for (int k = 0; k < d; k++)
    {
      whole *= (kv.first[k] <= 1) ? 1 : int64_t(1) << (kv.first[k] - 1);
      if (kv.first[k] > 0)
      {
        key = kv.first;
        key[k]--;
        if (levels.count(key) == 0)
          return false;
      }
    }
    if (kv.second != whole)
      return false;
  }
  return true;
}

int64_t fibre_lanes(akm_matrix_s const &m, std::vector<gk_lists> const &lists,
                    std::vector<std::vector<int>> const &term_act)
{
  const program prog(m.T, term_act);
  // half of the connections lie on each side of the diagonal
  int64_t steps = 0;
  for (auto const &p : prog.prods)
    steps += static_cast<int64_t>(lists[p.k].cell.size()) / (p.fill == gk_full ? 1 : 2);
  return steps * m.N;
}

int build_fibre_plan(akm_matrix_s const &m, int64_t active_cells, int64_t cells, const int *elem,
                     std::vector<gk_lists> const &lists,
                     std::vector<std::vector<int>> const &term_act,
                     std::vector<int> const &c1_diag, fibre_plan &plan)
{
  const int d = m.d, n = m.n, N = static_cast<int>(m.N);
  const program prog(m.T, term_act);
  // lanes share a workgroup's LDS by slot; wider tensors and larger blocks
  // take one workgroup per cell and 256 entries.  Workgroups of 256 threads start sooner
  // (d = 2, n = 2, level 5: 3.2 us an apply against 3.6 with 512 and 5.0 with
  // 1024); from 65 entries on a cell's list needs the slots of 1024 (d = 4,
  // n = 3, level 5: 9.4 us against 10.9 with 256 or 512)
  plan.slots_of_lanes = n <= 4 && N <= 1024;
  plan.tpb = N <= 64 ? 256 : 1024;
  plan.nslot = plan.slots_of_lanes ? plan.tpb / N : 1;
  plan.vectors = prog.vectors;
  plan.identities = prog.identities;
  plan.ntab = static_cast<int>(prog.tables.size());
  plan.nconn = m.nconn;
  plan.M = m.M;
  plan.stride = cells * N;
  const int64_t blocks = int64_t(plan.nconn) + 2 * plan.M; // of one table
  if (blocks * plan.ntab >= (int64_t(1) << 31) - 1 || cells >= (int64_t(1) << 31))
    return set_error(AKM_ERR_UNSUPPORTED, "fibre plan: factor tables too large");
  const int zero_block = static_cast<int>(blocks * plan.ntab);

  std::vector<int> stride(d, 1);
  for (int k = d - 2; k >= 0; k--)
    stride[k] = stride[k + 1] * n;
  std::vector<unsigned> magic(d);
  for (int k = 0; k < d; k++)
    magic[k] = (stride[k] == 1)
                   ? 0
                   : static_cast<unsigned>(((uint64_t(1) << 32) + stride[k] - 1) / stride[k]);

  // A job is one cell of one output vector.  cut() deals its products'
  // connections out in pieces: piece(product, list, from, to, connections,
  // first of a slot) for every piece in order.
  const int S = plan.nslot;
  struct output
  {
    int vec; // as fl_slot_rec
    std::vector<product> prods;
  };
  struct job
  {
    const output *out;
    int cell;
    int slots, more; // slots; pieces beyond the slots' first ones
    int length;      // connections
    int64_t slot0, piece0;
  };
  auto cut = [&](output const &out, int c, auto &&piece) -> int64_t {
    int64_t total = 0, whole = 0; // connections; slots with one piece each
    for (product const &p : out.prods)
    {
      int lo, hi;
      fill_range(lists[p.k], c, p.fill, lo, hi);
      total += hi - lo;
      whole += (hi - lo + fl_piece - 1) / fl_piece;
    }
    // slots of equal length when one-piece slots do not fit
    const bool split = whole <= S;
    const int64_t target = split ? fl_piece : (total + S - 1) / S;
    int64_t room = 0;
    for (product const &p : out.prods)
    {
      gk_lists const &l = lists[p.k];
      int lo, hi;
      fill_range(l, c, p.fill, lo, hi);
      if (split)
        room = 0; // pieces do not share slots
      while (lo < hi)
      {
        const bool fresh = room == 0;
        if (fresh)
          room = target;
        const int from = lo;
        int len = 0;
        if (p.in != 0 || active_cells == cells)
        {
          len = static_cast<int>(std::min<int64_t>({hi - lo, fl_piece, room}));
          lo += len;
        }
        else
          // cells the input does not hold are zero
          for (; lo < hi && len < fl_piece && len < room; lo++)
            len += (l.cell[lo] < active_cells) ? 1 : 0;
        piece(p, l, from, lo, len, fresh);
        room -= len;
      }
    }
    return total;
  };

  // stage by stage: every job's size, then the jobs of many slots first, then
  // long ones (a wavefront's pieces are alike and the long jobs start early),
  // which gives every record its place
  const int nstages = std::max(prog.stages, 1);
  std::vector<job> jobs; // in their order in the plan
  std::deque<output> outs;
  std::vector<size_t> stage_end(nstages);
  int64_t nslots = 0, npieces = 0;
  for (int st = 0; st < nstages; st++)
  {
    std::map<int, std::vector<product>> by_out;
    for (product const &p : prog.prods)
      if (p.stage == st)
        by_out[p.out].push_back(p);
    if (st + 1 == nstages)
      by_out[-1]; // y is always written
    std::vector<job> made;
    for (auto &ov : by_out)
    {
      // products of one dimension together: a slot's rounds are few
      std::stable_sort(ov.second.begin(), ov.second.end(),
                       [](product const &u, product const &v) { return u.k < v.k; });
      const int64_t ncell = (ov.first < 0) ? active_cells : cells;
      outs.push_back({ov.first < 0 ? -1 : ov.first - 1, std::move(ov.second)});
      output const &out = outs.back();
      made.reserve(made.size() + ncell);
      for (int64_t c = 0; c < ncell; c++)
      {
        job jb{&out, static_cast<int>(c), 0, 0, 0, 0, 0};
        const int64_t total =
            cut(out, jb.cell,
                [&](product const &, gk_lists const &, int, int, int, bool fresh) {
                  (fresh ? jb.slots : jb.more)++;
                });
        jb.slots = std::max(jb.slots, 1);
        jb.length = static_cast<int>(std::min<int64_t>(total, 1 << 30));
        made.push_back(jb);
      }
    }
    int most = 0, longest = 0;
    for (job const &jb : made)
    {
      most = std::max(most, jb.slots);
      longest = std::max(longest, jb.length);
    }
    int bits = 1; // of a length
    while (longest >> bits != 0)
      bits++;
    std::vector<uint64_t> keys(made.size());
    for (size_t i = 0; i < made.size(); i++)
      keys[i] = static_cast<uint64_t>(most - made[i].slots) << bits |
                static_cast<uint64_t>(longest - made[i].length);
    int all = bits + 1;
    while (most >> (all - bits) != 0)
      all++;
    std::vector<int> order;
    radix_order(keys, all, order);
    fibre_plan::stage rec;
    rec.first_group = static_cast<int>(nslots / S);
    for (int i : order)
    {
      job &jb = made[i];
      if (nslots % S != 0 && S - nslots % S < jb.slots)
        nslots += S - nslots % S;
      jb.slot0 = nslots;
      jb.piece0 = npieces;
      nslots += jb.slots;
      npieces += jb.more;
      jobs.push_back(jb);
    }
    nslots = (nslots + S - 1) / S * S;
    rec.groups = static_cast<int>(nslots / S) - rec.first_group;
    plan.stages.push_back(rec);
    stage_end[st] = jobs.size();
  }
  if (nslots > (int64_t(1) << 28) || npieces > (int64_t(1) << 28))
    return set_error(AKM_ERR_UNSUPPORTED, "fibre plan: too many slots");

  // the records, each written once where it stays
  std::unique_ptr<fl_slot_rec[]> slots(new fl_slot_rec[nslots]);
  std::unique_ptr<fl_piece_rec[]> pieces(new fl_piece_rec[npieces]);
  auto write = [&](fl_piece_rec &r, product const &p, int cell, int len) {
    r.in = p.in;
    r.stride = stride[p.k];
    r.magic = magic[p.k];
    r.len = len | (1 << 16);
    const int2 rest = make_int2(p.in == 0 && cell >= active_cells ? 0 : cell, zero_block);
    for (int u = len; u < fl_piece; u++)
      r.entry[u] = rest;
  };
  auto fill_job = [&](job const &jb) {
    fl_slot_rec *sr = slots.get() + jb.slot0 - 1;
    fl_piece_rec *more = pieces.get() + jb.piece0, *before = nullptr;
    int rank = 0;
    auto open_slot = [&] {
      sr++;
      sr->cell = jb.cell;
      sr->group = rank++ | jb.slots << 16;
      sr->vec = jb.out->vec;
      sr->more = sr->next = 0;
      sr->rounds = 1;
      sr->pad[0] = sr->pad[1] = 0;
    };
    cut(*jb.out, jb.cell,
        [&](product const &p, gk_lists const &l, int from, int to, int len, bool fresh) {
          if (fresh)
            open_slot();
          fl_piece_rec &r = fresh ? sr->p : *more;
          write(r, p, jb.cell, len);
          const bool all = p.in != 0 || active_cells == cells;
          int u = 0;
          for (int q = from; q < to; q++)
          {
            if (!all && l.cell[q] >= active_cells)
              continue;
            int b = l.q[q];
            if (q == l.diag[jb.cell] && p.fill != gk_full)
              b = plan.nconn + elem[int64_t(jb.cell) * d + p.k] +
                  (p.fill == gk_lower ? plan.M : 0);
            r.entry[u++] = make_int2(l.cell[q], static_cast<int>(p.table * blocks + b));
          }
          if (!fresh)
          {
            if (before->stride == r.stride)
              before->len &= 0xffff; // the same round goes on
            else
              sr->rounds++;
            if (sr->more++ == 0)
              sr->next = static_cast<int>(more - pieces.get());
            more++;
          }
          before = &r;
        });
    if (rank == 0)
    {
      open_slot();
      write(sr->p, product{0, 0, 0, gk_full, 0, 0}, jb.cell, 0);
    }
  };
  fl_slot_rec empty{};
  empty.cell = -1;
  int64_t done = 0; // slots written
  size_t at = 0;
  for (int st = 0; st < nstages; st++)
  {
    for (; at < stage_end[st]; at++)
    {
      for (; done < jobs[at].slot0; done++)
        slots[done] = empty;
      fill_job(jobs[at]);
      done = jobs[at].slot0 + jobs[at].slots;
    }
    const int64_t end = int64_t(plan.stages[st].first_group + plan.stages[st].groups) * S;
    for (; done < end; done++)
      slots[done] = empty;
  }
  for (int64_t g = 0; g < nslots; g += S)
  {
    int rounds = 1;
    for (int i = 0; i < S; i++)
      rounds = std::max(rounds, slots[g + i].rounds);
    if (rounds > 1)
      for (int i = 0; i < S; i++)
        slots[g + i].rounds = rounds;
  }

  std::vector<int> ptr(1, 0), src;
  for (auto const &t : prog.tables)
  {
    for (auto const &pr : t)
      src.insert(src.end(), {pr.first, pr.second});
    ptr.push_back(static_cast<int>(src.size() / 2));
  }
  AKM_TRY(plan.slots.upload(reinterpret_cast<const int4 *>(slots.get()), nslots * 7, m.stream));
  AKM_TRY(plan.pieces.upload(reinterpret_cast<const int4 *>(pieces.get()), npieces * 5, m.stream));
  // one array: tab_ptr, tab_src, connect_1d's diagonal positions
  std::vector<int> small = ptr;
  plan.src0 = static_cast<int>(small.size());
  small.insert(small.end(), src.begin(), src.end());
  plan.diag0 = static_cast<int>(small.size());
  small.insert(small.end(), c1_diag.begin(), c1_diag.end());
  AKM_TRY(plan.tab_def.upload(small.data(), int64_t(small.size()), m.stream));
  AKM_TRY(plan.work.allocate(int64_t(plan.vectors) * plan.stride * int64_t(m.esize)));
  AKM_TRY(plan.tab.allocate((blocks * plan.ntab + 1) * n * n * int64_t(m.esize)));
  plan.tab_valid = false;
  plan.built = true;
  return AKM_SUCCESS;
}

//! Rebuilds the factor tables when vA changed since they were built.
template<typename P>
static int fibre_tables(akm_matrix_s const &m, fibre_plan &plan, hipStream_t stream)
{
  if (plan.tab_valid && plan.stamp == m.vA_stamp)
    return AKM_SUCCESS;
  const int nn = m.n * m.n;
  const int64_t count = int64_t(plan.nconn + 2 * plan.M) * nn * plan.ntab + nn;
  const int64_t blocks = std::min<int64_t>((count + 255) / 256, 4096);
  fl_tables<P><<<static_cast<unsigned>(blocks), 256, 0, stream>>>(
      reinterpret_cast<const P *>(m.vA.data()), plan.tab_def.data(),
      plan.tab_def.data() + plan.src0, plan.tab_def.data() + plan.diag0, plan.ntab, plan.nconn, plan.M, m.n, m.d, m.T,
      reinterpret_cast<P *>(plan.tab.data()));
  plan.stamp = m.vA_stamp;
  plan.tab_valid = true;
  return check_launch("fibre tables");
}

//! The plan's part of the kernel arguments.
template<typename P, typename X>
static fl_args<P, X> fibre_args(akm_matrix_s const &m, fibre_plan const &plan)
{
  fl_args<P, X> a{};
  a.slots = plan.slots.data();
  a.pieces = plan.pieces.data();
  a.tab = reinterpret_cast<const P *>(plan.tab.data());
  a.n = m.n;
  a.N = static_cast<int>(m.N);
  a.nslot = plan.nslot;
  a.stride = plan.stride;
  a.work = reinterpret_cast<P *>(plan.work.data());
  a.identities = plan.identities;
  return a;
}

template<typename P, typename X>
static int launch_stage(akm_matrix_s const &m, fibre_plan const &plan,
                        fibre_plan::stage const &st, fl_args<P, X> const &a)
{
  const dim3 grid(static_cast<unsigned>(st.groups)), tpb(static_cast<unsigned>(plan.tpb));
  const size_t lds = sizeof(P) * plan.tpb * m.n;
  auto go = [&](auto small, auto large) {
    if (plan.tpb == 256)
      small<<<grid, tpb, lds, m.stream>>>(a, st.first_group);
    else
      large<<<grid, tpb, lds, m.stream>>>(a, st.first_group);
    return check_launch("fibre stage");
  };
  if (m.n == 1)
    return go(fl_stage<P, 1, 256, X>, fl_stage<P, 1, 256, X>); // one lane a slot
  if (m.n == 2)
    return go(fl_stage<P, 2, 256, X>, fl_stage<P, 2, 1024, X>);
  if (m.n == 3)
    return go(fl_stage<P, 3, 256, X>, fl_stage<P, 3, 1024, X>);
  return go(fl_stage<P, 4, 256, X>, fl_stage<P, 4, 1024, X>);
}

template<typename P>
int fibre_apply(akm_matrix_s &m, fibre_plan &plan, P alpha, const P *x, P beta, P *y, P gamma,
                const P *xg, const double *pc, double jdt)
{
  fl_args<P> a = fibre_args<P, P>(m, plan);
  a.x = x;
  a.y = y;
  a.xg = xg;
  a.pc = pc;
  a.jdt = jdt;
  a.alpha = alpha;
  a.beta = beta;
  a.gamma = gamma;
  for (auto const &st : plan.stages)
  {
    if (plan.slots_of_lanes)
    {
      AKM_TRY(launch_stage(m, plan, st, a));
      continue;
    }
    const dim3 grid(static_cast<unsigned>(st.groups),
                    static_cast<unsigned>((a.N + fl_any_width - 1) / fl_any_width));
    auto go = [&](auto small, auto large) {
      if (plan.tpb == 256)
        small<<<grid, 256, 0, m.stream>>>(a, st.first_group);
      else
        large<<<grid, 1024, 0, m.stream>>>(a, st.first_group);
    };
    if (a.n == 5)
      go(fl_stage_any<P, 5, 256>, fl_stage_any<P, 5, 1024>);
    else
      go(fl_stage_any<P, 0, 256>, fl_stage_any<P, 0, 1024>);
    AKM_TRY(check_launch("fibre stage"));
  }
  return AKM_SUCCESS;
}

int fibre_refresh(akm_matrix_s const &m, fibre_plan &plan, hipStream_t stream)
{
  return (m.prec == AKM_F64) ? fibre_tables<double>(m, plan, stream)
                             : fibre_tables<float>(m, plan, stream);
}

fibre_system fibre_batch_system(akm_matrix_s const &m, fibre_plan const &plan, double *V,
                                double *X, int64_t size, double dt)
{
  const fl_args<double> a = fibre_args<double, double>(m, plan);
  return fibre_system{a.slots, a.pieces, a.tab, V, X, size, dt, a.n, a.N, a.nslot, a.identities};
}

int launch_fibre_batch(int tpb, int groups, const fibre_system *fs, const int2 *items,
                       const int *jcol, int joff, int limit, const int *active, int phase,
                       hipStream_t stream)
{
  if (groups <= 0)
    return AKM_SUCCESS;
  const size_t lds = sizeof(double) * tpb * 4;
  if (tpb == 256)
    fl_batch<256><<<groups, 256, lds, stream>>>(fs, items, jcol, joff, limit, active, phase);
  else
    fl_batch<1024><<<groups, 1024, lds, stream>>>(fs, items, jcol, joff, limit, active, phase);
  return check_launch("batched fibre walk");
}

bool fibre_apply_between(akm_matrix_s &m, fibre_plan &plan, const double *v, double c, double *w)
{
  if (!plan.built || !plan.slots_of_lanes || plan.stages.size() != 1 || plan.vectors != 0)
    return false;
  fl_args<float, double> a = fibre_args<float, double>(m, plan);
  a.x = v;
  a.y = w;
  a.xg = v;
  a.between = c;
  return launch_stage(m, plan, plan.stages[0], a) == AKM_SUCCESS;
}

template int fibre_apply<double>(akm_matrix_s &, fibre_plan &, double, const double *, double,
                                 double *, double, const double *, const double *, double);
template int fibre_apply<float>(akm_matrix_s &, fibre_plan &, float, const float *, float,
                                float *, float, const float *, const double *, double);
} // namespace akm
