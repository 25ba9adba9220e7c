// Learned right preconditioner of the flexible GMRES: a per-cell MLP.
//
// For every grid cell c with residual block r_c (the cell's n^d
// coefficients) and norm s = |r_c|, the network reads
//   x = [ r_c / s , f_c , 0 pad ]            (K1 = roundup16(n^d + d) inputs)
// where f_c holds one feature per dimension: level + (position + 1/2) /
// cells-of-the-level, divided by max_level + 1.  Two hidden layers of H ReLU
// units and a linear output o (n^d values, padded to N3 = roundup16(n^d))
// give the correction
//   z_c = r_c + s * o(x)
// so an untrained network (zero output layer) is the identity.  Training
// fits o to (e_c - r_c) / s on (residual, correction) pairs of the plain
// solver, e = (I - dt A)^-1 r, with the mean squared error.
//
// Parameters live as one flat FP32 array
//   [ W1 (H x K1) | b1 (H) | W2 (H x H) | b2 (H) | W3 (N3 x H) | b3 (N3) ]
// with every W row-major (output x input).  Training runs in FP32 on the
// matrix cores (v_mfma_f32_16x16x4_f32: FP32 products and sums): one kernel
// takes 16 samples through the whole forward and backward chain with their
// activations in LDS, a second forms every weight and bias gradient, a third
// adds its row parts.  The preconditioner itself runs on BF16 copies of W1..W3
// with v_mfma_f32_16x16x32_bf16 (FP32 accumulation), eight wavefronts per 16 to
// 64 cells, activations in LDS.
#include "precond.hpp"

#include <algorithm>
#include <cmath>
#include <memory>
#include <numeric>
#include <random>
#include <vector>

namespace akm
{
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int mc_rows = 16;    // samples per workgroup of the chain kernel
constexpr int mc_waves = 16;   // its wavefronts, which share the output columns
constexpr int mc_threads = mc_waves * 64;
constexpr int wg_tile = 32;    // weight-gradient tile (outputs x inputs)
constexpr int wg_threads = 256; // its four wavefronts split the rows
constexpr int wg_max_parts = 16;

//! Barrier that orders LDS accesses only: a full one would also wait for the
//! activations' stores to memory, which no wavefront of the kernel reads.
__device__ __forceinline__ void mlp_lds_barrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

//! 16 samples x 16 outputs from j0 on: in (16 x K, LDS, rows ldi apart) times
//! W^T (outputs x inputs, BACK = false) or times W (BACK = true: inputs x
//! outputs).  Operands of v_mfma_f32_16x16x4_f32: lane l holds
//! A[l % 16][l / 16] and B[l / 16][l % 16], and gets D[4 (l / 16) + i][l % 16].
//! The sum over k may run in any order, so lane group g takes k = 16 b + 4 g
//! + i in step i: four consecutive inputs, one 16-byte read.  The four steps
//! have a sum each, added at the end: shorter chains of rounded sums, and no
//! step waits for the one before.
template<bool BACK>
__device__ __forceinline__ f32x4 mlp_tile(const float *in, int ldi, int K, const float *W,
                                          int ldw, int j0)
{
  // blocks of 16 inputs read ahead: with two a row's 128-byte lines are read
  // whole; three and four are slower (35 us, as below), as more rows' lines
  // contend for the same sets of the first-level cache
  constexpr int U = 2;
  f32x4 acc[4] = {};
  const int lane = threadIdx.x % 64, row = lane % 16, g = lane / 16;
  const float *arow = in + row * ldi + 4 * g;
  const float *w = BACK ? W + int64_t(4 * g) * ldw + j0 + row
                        : W + int64_t(j0 + row) * ldw + 4 * g;
  // all reads of U blocks in flight; those past K repeat the last block's
  auto read = [&](int k0, f32x4 (&b)[U]) {
#pragma unroll
    for (int u = 0; u < U; u++)
    {
      const int k = min(k0 + 16 * u, K - 16);
      if constexpr (BACK)
      {
#pragma unroll
        for (int i = 0; i < 4; i++)
          b[u][i] = w[int64_t(k + i) * ldw];
      }
      else
        b[u] = *reinterpret_cast<const f32x4 *>(w + k);
    }
  };
  f32x4 cur[U], next[U];
  read(0, cur);
  for (int k0 = 0; k0 < K; k0 += 16 * U)
  {
    read(k0 + 16 * U, next);
    // the scheduler would move each read to its use
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (k0 + 16 * u < K)
      {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(arow + k0 + 16 * u);
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], cur[u][i], acc[i], 0, 0, 0);
      }
#pragma unroll
    for (int u = 0; u < U; u++)
      cur[u] = next[u];
  }
  return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}

//! One layer for the workgroup's 16 samples: put(sample, output, values of
//! this and the next three samples) for every output of J (a multiple of 16).
//! Wavefronts take every mc_waves-th tile of 16 outputs.
template<bool BACK, typename Put>
__device__ __forceinline__ void mlp_layer(const float *in, int ldi, int K, const float *W,
                                          int ldw, int J, Put &&put)
{
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma nounroll
  for (int j0 = 16 * wave; j0 < J; j0 += 16 * mc_waves)
    put(4 * (lane / 16), j0 + lane % 16, mlp_tile<BACK>(in, ldi, K, W, ldw, j0));
}

//! Shapes, parameters and buffers of a training pass.
struct mlp_pass
{
  int64_t rows;
  int N, N3, K1, H;
  const float *W1, *b1, *W2, *b2, *W3, *b3;
  const float *X, *T;
  float *H1, *H2, *O, *dO, *dH2, *dH1;
  float scale;     // of the output gradient
  double *partial; // per workgroup: sum of (O - T)^2
};

//! 16 samples through the layers (H1, H2, O to memory), and with BACK back
//! again: dO = scale (O - T) on the first N of N3 outputs, dH2, dH1.
//! What bounds it: the weights' way from L2, which every workgroup reads whole;
//! with the products taken out the 256 x 256 layer takes as long (10 us), with
//! the reads taken out half as long, and its matrix-core time is 3.6 us.
//! 1024 samples of 80 -> 256 -> 256 -> 64 take 32 us (64 workgroups),
//! 32768 take 235 us; with 8 wavefronts of two tiles each 37 and 311 us.
//! Separate tiled products took 12-34 us for each of the layers (64 x 64
//! tiles leave most of the chip idle).
//! LDS: 16 x (K1 + 2 H + N3 + 16) floats, rows 4 floats apart beyond their
//! length so that 16-byte reads of 16 rows spread over the banks.
template<bool BACK>
__global__ void __launch_bounds__(mc_threads) mlp_chain(mlp_pass p)
{
  extern __shared__ __align__(16) float mc_lds[];
  __shared__ double sh[mc_waves];
  const int ldx = p.K1 + 4, ldh = p.H + 4, ldo = p.N3 + 4;
  float *Xs = mc_lds, *A1 = Xs + mc_rows * ldx, *A2 = A1 + mc_rows * ldh,
        *Os = A2 + mc_rows * ldh;
  const int64_t r0 = int64_t(blockIdx.x) * mc_rows;
  const int live = static_cast<int>(min(int64_t(mc_rows), p.rows - r0));
  for (int e = threadIdx.x; e < mc_rows * p.K1; e += mc_threads)
  {
    const int r = e / p.K1, i = e - r * p.K1;
    Xs[r * ldx + i] = (r < live) ? p.X[(r0 + r) * p.K1 + i] : 0.0f;
  }
  mlp_lds_barrier();
  double sq = 0;
  auto hidden = [&](const float *in, int K, const float *W, const float *bias, float *keep,
                    float *out) {
    mlp_layer<false>(in, K + 4, K, W, K, p.H, [&](int r, int j, f32x4 v) {
      const float b = bias[j];
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const float x = fmaxf(v[i] + b, 0.0f);
        keep[(r + i) * ldh + j] = x;
        if (r + i < live)
          out[(r0 + r + i) * p.H + j] = x;
      }
    });
    mlp_lds_barrier();
  };
  hidden(Xs, p.K1, p.W1, p.b1, A1, p.H1);
  hidden(A1, p.H, p.W2, p.b2, A2, p.H2);
  mlp_layer<false>(A2, ldh, p.H, p.W3, p.H, p.N3, [&](int r, int j, f32x4 v) {
    const float b = p.b3[j];
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
      float x = v[i] + b;
      if constexpr (BACK)
      {
        float grad = 0.0f;
        if (r + i < live && j < p.N)
        {
          const float diff = x - p.T[(r0 + r + i) * p.N3 + j];
          sq += double(diff) * double(diff);
          grad = p.scale * diff;
        }
        Os[(r + i) * ldo + j] = grad;
        x = grad;
      }
      if (r + i < live)
        (BACK ? p.dO : p.O)[(r0 + r + i) * p.N3 + j] = x;
    }
  });
  if constexpr (BACK)
  {
    mlp_lds_barrier();
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      sq += __shfl_xor(sq, off);
    if (threadIdx.x % 64 == 0)
      sh[threadIdx.x / 64] = sq;
    // the masks are the activations, which their gradients replace in LDS
    auto back = [&](const float *in, int K, const float *W, float *mask, float *out) {
      mlp_layer<true>(in, K + 4, K, W, p.H, p.H, [&](int r, int j, f32x4 v) {
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
          const float x = (mask[(r + i) * ldh + j] > 0.0f) ? v[i] : 0.0f;
          mask[(r + i) * ldh + j] = x;
          if (r + i < live)
            out[(r0 + r + i) * p.H + j] = x;
        }
      });
      mlp_lds_barrier();
    };
    back(Os, p.N3, p.W3, A2, p.dH2);
    back(A2, p.H, p.W2, A1, p.dH1);
    if (threadIdx.x == 0)
    {
      double t = 0;
      for (int w = 0; w < mc_waves; w++)
        t += sh[w];
      p.partial[blockIdx.x] = t;
    }
  }
}

//! One weight gradient dW = G^T Y (G: rows x M, Y: rows x C, dW: M x C) and
//! its bias gradient (the column sums of G), as a range of tiles.
struct wg_layer
{
  const float *G, *Y;
  int M, C;
  int64_t oW, ob; // offsets in the flat gradient
  int tile0;      // first tile of the layer
};
struct wg_args
{
  wg_layer layer[3];
  int64_t rows, chunk; // rows per part
  int64_t stride;      // values of one part
  float *out;          // part z of the gradient at out + z * stride
};

//! A 32 x 32 tile of one layer's gradient over the rows of part blockIdx.y.
//! The four wavefronts take every fourth 16 rows and their sums meet in LDS
//! in wavefront order.
__global__ void __launch_bounds__(wg_threads) mlp_weight_grad(wg_args a)
{
  __shared__ float red[4][wg_tile][wg_tile + 1];
  __shared__ float bred[4][wg_tile];
  const int tile = blockIdx.x;
  const int li = (tile >= a.layer[2].tile0) ? 2 : (tile >= a.layer[1].tile0 ? 1 : 0);
  const wg_layer L = a.layer[li];
  const int ctiles = (L.C + wg_tile - 1) / wg_tile;
  const int m0 = (tile - L.tile0) / ctiles * wg_tile, c0 = (tile - L.tile0) % ctiles * wg_tile;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, col = lane % 16, g = lane / 16;
  const int64_t b0 = blockIdx.y * a.chunk, b1 = min(a.rows, b0 + a.chunk);
  f32x4 acc[2][2] = {};
  float bias[2] = {0.0f, 0.0f};
  // outputs and inputs past the layer's read its first ones and are dropped
  int mi[2], ci[2];
#pragma unroll
  for (int t = 0; t < 2; t++)
  {
    mi[t] = (m0 + 16 * t < L.M) ? m0 + 16 * t + col : col;
    ci[t] = (c0 + 16 * t < L.C) ? c0 + 16 * t + col : col;
  }
  // two blocks of 16 rows a round, all reads in flight
  constexpr int U = 2;
  for (int64_t b = b0 + 16 * wave; b < b1; b += 64 * U)
  {
    float gv[U][2][4], yv[U][2][4];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const int64_t r = b + 64 * u + 4 * g + i;
        const int64_t rr = (r < b1) ? r : b0;
#pragma unroll
        for (int t = 0; t < 2; t++)
        {
          gv[u][t][i] = L.G[rr * L.M + mi[t]];
          yv[u][t][i] = L.Y[rr * L.C + ci[t]];
        }
      }
    __builtin_amdgcn_sched_barrier(0); // the reads stay ahead of the products
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const bool live = b + 64 * u + 4 * g + i < b1;
#pragma unroll
        for (int t = 0; t < 2; t++)
        {
          gv[u][t][i] = live ? gv[u][t][i] : 0.0f;
          yv[u][t][i] = live ? yv[u][t][i] : 0.0f;
          bias[t] += gv[u][t][i];
        }
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int v = 0; v < 2; v++)
            acc[t][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(gv[u][t][i], yv[u][v][i], acc[t][v],
                                                             0, 0, 0);
      }
  }
#pragma unroll
  for (int t = 0; t < 2; t++)
  {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        red[wave][16 * t + 4 * g + i][16 * u + col] = acc[t][u][i];
    bias[t] += __shfl_xor(bias[t], 16);
    bias[t] += __shfl_xor(bias[t], 32);
    if (g == 0)
      bred[wave][16 * t + col] = bias[t];
  }
  __syncthreads();
  float *out = a.out + blockIdx.y * a.stride;
  for (int e = threadIdx.x; e < wg_tile * wg_tile; e += wg_threads)
  {
    const int m = e / wg_tile, c = e % wg_tile;
    if (m0 + m < L.M && c0 + c < L.C)
      out[L.oW + int64_t(m0 + m) * L.C + c0 + c] =
          (red[0][m][c] + red[1][m][c]) + (red[2][m][c] + red[3][m][c]);
  }
  if (c0 == 0 && threadIdx.x < wg_tile && m0 + static_cast<int>(threadIdx.x) < L.M)
  {
    const int m = threadIdx.x;
    out[L.ob + m0 + m] = (bred[0][m] + bred[1][m]) + (bred[2][m] + bred[3][m]);
  }
}

//! grad[e] = sum over z < parts of part[z*count + e] in order (parts = 1: grad
//! is already complete); the last block adds the `losses` partial losses into
//! loss[0] (accumulated if `accumulate`), in a fixed order, and stores it to
//! the host as well.
__global__ void __launch_bounds__(256)
mlp_sum_parts(int64_t count, int parts, const float *part, float *grad, int losses,
              const double *partial, double *loss, int accumulate, double *host_loss)
{
  __shared__ double sh[256];
  if (blockIdx.x + 1 == gridDim.x)
  {
    double s = 0;
    for (int i = threadIdx.x; i < losses; i += 256)
      s += partial[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1)
    {
      if (threadIdx.x < k)
        sh[threadIdx.x] += sh[threadIdx.x + k];
      __syncthreads();
    }
    if (threadIdx.x == 0)
    {
      const double total = accumulate ? loss[0] + sh[0] : sh[0];
      loss[0] = total;
      __hip_atomic_store(host_loss, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return;
  }
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < count; e += 256ll * (gridDim.x - 1))
  {
    float s = part[e];
    for (int z = 1; z < parts; z++)
      s += part[z * count + e];
    grad[e] = s;
  }
}

//! Adam (Kingma & Ba, 2015): m = b1 m + (1-b1) g, v = b2 v + (1-b2) g^2,
//! p -= lr * (m c1) / (sqrt(v c2) + eps) with the bias corrections
//! c1 = 1/(1-b1^t), c2 = 1/(1-b2^t).
__global__ void __launch_bounds__(256)
mlp_adam(int64_t count, float *p, const float *g, float *m, float *v, float lr, float b1,
         float b2, float eps, float c1, float c2)
{
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < count; i += 256ll * gridDim.x)
  {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
  }
}

//! Samples of the pairs: for vector q and cell c (sample q*cells + c),
//! X row = [r/s, features, 0], T row = [(e - r)/s, 0], s = |r_c|.
__global__ void __launch_bounds__(256)
mlp_make_samples(int64_t nvec, int64_t cells, int N, int d, int K1, int N3, const double *R,
                 const double *E, const float *feat, float *X, float *T)
{
  const int64_t total = nvec * cells;
  for (int64_t q = blockIdx.x * 256ll + threadIdx.x; q < total; q += 256ll * gridDim.x)
  {
    const int64_t c = q % cells;
    const double *r = R + q * N;
    const double *e = E + q * N;
    double s = 0;
    for (int i = 0; i < N; i++)
      s = fma(r[i], r[i], s);
    s = sqrt(s);
    const double inv = (s > 0.0) ? 1.0 / s : 0.0;
    float *x = X + q * K1;
    float *y = T + q * N3;
    for (int i = 0; i < N; i++)
    {
      x[i] = static_cast<float>(r[i] * inv);
      y[i] = static_cast<float>((e[i] - r[i]) * inv);
    }
    for (int k = 0; k < d; k++)
      x[N + k] = feat[c * d + k];
    for (int i = N + d; i < K1; i++)
      x[i] = 0.0f;
    for (int i = N; i < N3; i++)
      y[i] = 0.0f;
  }
}

//! Rows perm[base .. base+rows) of X and T into the batch buffers.
__global__ void __launch_bounds__(256)
mlp_gather(int rows, const int64_t *perm, int64_t base, int K1, int N3, const float *X,
           const float *T, float *Xb, float *Tb)
{
  const int r = blockIdx.x;
  if (r >= rows)
    return;
  const int64_t src = perm[base + r];
  for (int i = threadIdx.x; i < K1; i += 256)
    Xb[int64_t(r) * K1 + i] = X[src * K1 + i];
  for (int i = threadIdx.x; i < N3; i += 256)
    Tb[int64_t(r) * N3 + i] = T[src * N3 + i];
}

//! FP32 -> BF16, round to nearest even (bias-and-truncate on the bit
//! pattern); NaN stays a quiet NaN.
__device__ __forceinline__ unsigned short to_bf16(float f)
{
  unsigned int u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u)
    return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<unsigned short>(u >> 16);
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

//! BF16 copy of W (J x K, J a multiple of 16) in the order the matrix cores
//! take it: tiles of 16 outputs x 32 inputs (the last one filled with zeros),
//! and in a tile 8 inputs for each lane, so that a wavefront reads 1 KB in
//! one piece.  KB tiles along the inputs, J16 along the outputs; outputs past
//! J are zero.
__global__ void __launch_bounds__(256)
mlp_pack_bf16(int J, int K, int J16, int KB, const float *src, unsigned short *dst)
{
  const int count = J16 * KB * 512;
  for (int e = blockIdx.x * 256 + threadIdx.x; e < count; e += 256 * gridDim.x)
  {
    const int tile = e / 512, lane = e / 8 % 64;
    const int j = tile / KB * 16 + lane % 16, k = tile % KB * 32 + lane / 16 * 8 + e % 8;
    dst[e] = (j < J && k < K) ? to_bf16(src[int64_t(j) * K + k]) : 0;
  }
}

constexpr int ma_waves = 8; // wavefronts of a workgroup, which share the outputs

//! T tiles of 16 outputs (from tile jt on) x R tiles of 16 cells on the matrix
//! cores: W packed (see mlp_pack_bf16), in BF16 rows of KB * 32 inputs in LDS.
//! v_mfma_f32_16x16x32_bf16 with the outputs as rows: lane l gives
//! W[l % 16][8 (l / 16) .. +7] and in[8 (l / 16) .. +7][l % 16] and gets
//! outputs 4 (l / 16) .. +3 of cell l % 16.
template<int T, int R>
__device__ __forceinline__ void mfma_tiles(const unsigned short *in, int ldi, int KB,
                                           const unsigned short *W, int jt, f32x4 (&acc)[T][R])
{
  constexpr int U = 2; // input tiles read ahead
  const int lane = threadIdx.x % 64;
  const unsigned short *arow = in + lane % 16 * ldi + lane / 16 * 8;
  const unsigned short *w = W + int64_t(jt) * KB * 512 + lane * 8;
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int r = 0; r < R; r++)
      acc[t][r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto read = [&](int kb, bf16x8 (&b)[U][T]) {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < T; t++)
        b[u][t] = *reinterpret_cast<const bf16x8 *>(w + (t * KB + min(kb + u, KB - 1)) * 512);
  };
  bf16x8 cur[U][T], next[U][T];
  read(0, cur);
  for (int kb = 0; kb < KB; kb += U)
  {
    read(kb + U, next);
    // the scheduler would move each read to its use
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (kb + u < KB)
      {
        bf16x8 a[R];
#pragma unroll
        for (int r = 0; r < R; r++)
          a[r] = *reinterpret_cast<const bf16x8 *>(arow + 16 * r * ldi + (kb + u) * 32);
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
          for (int r = 0; r < R; r++)
            acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[u][t], a[r], acc[t][r], 0, 0, 0);
      }
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < T; t++)
        cur[u][t] = next[u][t];
  }
}

//! A hidden layer (ReLU) of the workgroup's 16 R cells: 2 JT tiles of outputs,
//! J of them real; the others come out as zero.
template<int R>
__device__ __forceinline__ void mfma_layer(const unsigned short *in, int ldi, int KB,
                                           const unsigned short *W, const float *bias, int J,
                                           int JT, unsigned short *out, int ldo)
{
  const int lane = threadIdx.x % 64;
  for (int p = threadIdx.x / 64; p < JT; p += ma_waves)
  {
    f32x4 acc[2][R];
    f32x4 b[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const int j = 32 * p + 16 * t + lane / 16 * 4 + i;
        b[t][i] = (j < J) ? bias[j] : 0.0f;
      }
    mfma_tiles<2, R>(in, ldi, KB, W, 2 * p, acc);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < R; r++)
      {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; i++)
          x[i] = fmaxf(acc[t][r][i] + b[t][i], 0.0f);
        *reinterpret_cast<bf16x4 *>(out + (16 * r + lane % 16) * ldo + 32 * p + 16 * t +
                                    lane / 16 * 4) = __builtin_convertvector(x, bf16x4);
      }
  }
}

//! z = v + s * o(x) per cell (see the file comment) for 16 R cells a
//! workgroup, eight wavefronts sharing the outputs of each layer.
//! What bounds it: latency, from layer to layer, of the weights' way from L2
//! (208 KB a workgroup, in 1 KB pieces); at 16172 cells of 64 values, 256
//! wide, matrix-core time is 1.4 us and memory time 4 us of its 16.  One
//! wavefront per 16 cells, reading the weights row by row in 8-byte pieces
//! with nothing in flight beside the product, took 71 us.
//! LDS: rows of lda (inputs, then the second layer) and ldh (first layer)
//! BF16 values, 16 bytes longer than their contents so that 16 rows spread
//! over the banks; the norms.
template<int R>
__global__ void __launch_bounds__(64 * ma_waves, 4)
mlp_apply_bf16(int64_t cells, int N, int d, int H, int N3, int KB1, int KBH, const double *v,
               double *z, const float *feat, const unsigned short *W1, const float *b1,
               const unsigned short *W2, const float *b2, const unsigned short *W3,
               const float *b3)
{
  constexpr int C = 16 * R, TPC = 64 * ma_waves / C; // cells; threads per cell
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int lda = 32 * max(KB1, KBH) + 8, ldh = 32 * KBH + 8;
  float *snorm = reinterpret_cast<float *>(lds_raw);
  unsigned short *A = reinterpret_cast<unsigned short *>(lds_raw + sizeof(float) * C);
  unsigned short *H1s = A + C * lda;
  const int64_t c0 = int64_t(blockIdx.x) * C;
  {
    const int m = threadIdx.x / TPC, sub = threadIdx.x % TPC;
    const int64_t c = c0 + m;
    const double *vc = v + c * N;
    double sq = 0;
    if (c < cells)
      for (int i = sub; i < N; i += TPC)
        sq = fma(vc[i], vc[i], sq);
#pragma unroll
    for (int off = 1; off < TPC; off <<= 1)
      sq += __shfl_xor(sq, off);
    const float s = static_cast<float>(sqrt(sq));
    if (sub == 0)
      snorm[m] = s;
    for (int i = sub; i < 32 * KB1; i += TPC)
    {
      float x = 0.0f;
      if (c < cells)
      {
        if (i < N)
          x = (s > 0.0f) ? static_cast<float>(vc[i] / double(s)) : 0.0f;
        else if (i < N + d)
          x = feat[c * d + (i - N)];
      }
      A[m * lda + i] = to_bf16(x);
    }
  }
  mlp_lds_barrier();
  mfma_layer<R>(A, lda, KB1, W1, b1, H, KBH, H1s, ldh);
  mlp_lds_barrier();
  mfma_layer<R>(H1s, ldh, KBH, W2, b2, H, KBH, A, lda);
  mlp_lds_barrier();
  // output layer, linear, straight to z
  constexpr int RO = (R > 1) ? 2 : 1;
  const int lane = threadIdx.x % 64;
  for (int u = threadIdx.x / 64; u < N3 / 16 * (R / RO); u += ma_waves)
  {
    const int jt = u / (R / RO), r0 = u % (R / RO) * RO;
    f32x4 acc[1][RO];
    mfma_tiles<1, RO>(A + 16 * r0 * lda, lda, KBH, W3, jt, acc);
#pragma unroll
    for (int r = 0; r < RO; r++)
    {
      const int m = 16 * (r0 + r) + lane % 16;
      const int64_t c = c0 + m;
      if (c >= cells)
        continue;
      const double s = snorm[m];
#pragma unroll
      for (int i = 0; i < 4; i++)
      {
        const int j = 16 * jt + lane / 16 * 4 + i;
        if (j < N)
          z[c * N + j] = v[c * N + j] + s * double(acc[0][r][i] + b3[j]);
      }
    }
  }
}

static int64_t round16(int64_t v) { return (v + 15) / 16 * 16; }

static int grid_for(int64_t count)
{
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((count + 255) / 256, 4096)));
}

} // namespace akm

using namespace akm;

struct akm_mlp_s final : akm_precond_s
{
  int d = 0, n = 0, N = 0, N3 = 0, K1 = 0, H = 0;
  int64_t cells = 0;
  int max_level = 0;
  int64_t oW1 = 0, ob1 = 0, oW2 = 0, ob2 = 0, oW3 = 0, ob3 = 0, num_params = 0;
  dev_buffer<float> params, grad, adam_m, adam_v, feat;
  dev_buffer<unsigned short> wbf; // W1 | W2 | W3 in BF16 tiles
  bool bf16_current = false;
  int64_t adam_t = 0;
  // batch buffers (sized for `batch` rows)
  int batch = 0;
  dev_buffer<float> Xb, Tb, H1, H2, dO, dH2, dH1;
  dev_buffer<float> parts; // row parts of the gradient
  dev_buffer<double> partial, loss;
  double *host_loss = nullptr; // pinned copy of loss[0]
  hipStream_t stream = nullptr;

  ~akm_mlp_s() override
  {
    if (host_loss != nullptr)
      (void)hipHostFree(host_loss);
  }

  int64_t size() const override { return cells * N; }

  static int chain_groups(int B) { return (B + mc_rows - 1) / mc_rows; }
  //! Row parts of the weight gradients: 128 rows each, at most wg_max_parts.
  static int row_parts(int B) { return std::clamp(B / 128, 1, wg_max_parts); }

  int ensure_batch(int B)
  {
    if (B <= batch)
      return AKM_SUCCESS;
    batch = 0; // nothing to rely on until everything is there
    AKM_TRY(Xb.allocate(int64_t(B) * K1));
    AKM_TRY(Tb.allocate(int64_t(B) * N3));
    AKM_TRY(H1.allocate(int64_t(B) * H));
    AKM_TRY(H2.allocate(int64_t(B) * H));
    AKM_TRY(dO.allocate(int64_t(B) * N3));
    AKM_TRY(dH2.allocate(int64_t(B) * H));
    AKM_TRY(dH1.allocate(int64_t(B) * H));
    AKM_TRY(partial.allocate(chain_groups(B)));
    AKM_TRY(loss.allocate(2));
    if (host_loss == nullptr)
      AKM_HIP(hipHostMalloc(reinterpret_cast<void **>(&host_loss), sizeof(double),
                            hipHostMallocDefault));
    AKM_TRY(parts.allocate(row_parts(B) * num_params));
    batch = B;
    return AKM_SUCCESS;
  }

  //! The chain kernel on B rows of X (and T with BACK; O without).
  template<bool BACK>
  int chain(hipStream_t s, int B, const float *X, const float *T, float *O)
  {
    const float *p = params.data();
    mlp_pass a{};
    a.rows = B;
    a.N = N;
    a.N3 = N3;
    a.K1 = K1;
    a.H = H;
    a.W1 = p + oW1;
    a.b1 = p + ob1;
    a.W2 = p + oW2;
    a.b2 = p + ob2;
    a.W3 = p + oW3;
    a.b3 = p + ob3;
    a.X = X;
    a.T = T;
    a.H1 = H1.data();
    a.H2 = H2.data();
    a.O = O;
    a.dO = dO.data();
    a.dH2 = dH2.data();
    a.dH1 = dH1.data();
    a.scale = 2.0f / (float(B) * float(N));
    a.partial = partial.data();
    const size_t lds = sizeof(float) * mc_rows * size_t(K1 + 2 * H + N3 + 16);
    if (lds > 64 * 1024)
      AKM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(mlp_chain<BACK>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(lds)));
    mlp_chain<BACK><<<chain_groups(B), mc_threads, lds, s>>>(a);
    return check_launch("mlp layers");
  }

  //! FP32 forward of B rows of X into O (B x N3).
  int forward(hipStream_t s, int B, const float *X, float *O)
  {
    return chain<false>(s, B, X, nullptr, O);
  }

  //! Forward and backward of B rows: loss (squared error over B rows and N
  //! outputs) into loss[0] (accumulated if `accumulate`) and the gradient of
  //! every parameter into `out`.
  int gradients(hipStream_t s, int B, const float *X, const float *T, int accumulate, float *out)
  {
    AKM_TRY(chain<true>(s, B, X, T, nullptr));
    const int np = row_parts(B);
    wg_args a{};
    auto tiles = [](int M, int C) {
      return ((M + wg_tile - 1) / wg_tile) * ((C + wg_tile - 1) / wg_tile);
    };
    a.layer[0] = wg_layer{dH2.data(), H1.data(), H, H, oW2, ob2, 0};
    a.layer[1] = wg_layer{dH1.data(), X, H, K1, oW1, ob1, tiles(H, H)};
    a.layer[2] = wg_layer{dO.data(), H2.data(), N3, H, oW3, ob3, tiles(H, H) + tiles(H, K1)};
    a.rows = B;
    a.chunk = ((B + np - 1) / np + 15) / 16 * 16;
    a.stride = num_params;
    a.out = (np == 1) ? out : parts.data();
    mlp_weight_grad<<<dim3(a.layer[2].tile0 + tiles(N3, H), np), wg_threads, 0, s>>>(a);
    AKM_TRY(check_launch("mlp weight gradients"));
    const int blocks = (np == 1) ? 0 : grid_for(num_params);
    mlp_sum_parts<<<blocks + 1, 256, 0, s>>>(num_params, np, parts.data(), out, chain_groups(B),
                                             partial.data(), loss.data(), accumulate, host_loss);
    return check_launch("mlp gradients");
  }

  int adam(hipStream_t s, const float *g, float lr)
  {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    ++adam_t;
    const float c1 = static_cast<float>(1.0 / (1.0 - std::pow(double(b1), double(adam_t))));
    const float c2 = static_cast<float>(1.0 / (1.0 - std::pow(double(b2), double(adam_t))));
    mlp_adam<<<grid_for(num_params), 256, 0, s>>>(num_params, params.data(), g, adam_m.data(),
                                                  adam_v.data(), lr, b1, b2, eps, c1, c2);
    bf16_current = false;
    return check_launch("mlp adam");
  }

  int refresh_bf16(hipStream_t s)
  {
    if (bf16_current)
      return AKM_SUCCESS;
    const float *p = params.data();
    unsigned short *w = wbf.data();
    const int kb1 = kb(K1), kbh = kb(H);
    mlp_pack_bf16<<<grid_for(packed(2 * kbh, kb1)), 256, 0, s>>>(H, K1, 2 * kbh, kb1, p + oW1, w);
    w += packed(2 * kbh, kb1);
    mlp_pack_bf16<<<grid_for(packed(2 * kbh, kbh)), 256, 0, s>>>(H, H, 2 * kbh, kbh, p + oW2, w);
    w += packed(2 * kbh, kbh);
    mlp_pack_bf16<<<grid_for(packed(N3 / 16, kbh)), 256, 0, s>>>(N3, H, N3 / 16, kbh, p + oW3, w);
    AKM_TRY(check_launch("mlp bf16 weights"));
    bf16_current = true;
    return AKM_SUCCESS;
  }

  //! Tiles of 32 inputs, and values of a packed layer.
  static int kb(int K) { return (K + 31) / 32; }
  static int64_t packed(int J16, int KB) { return int64_t(J16) * KB * 512; }
  int64_t packed_weights() const
  {
    return packed(2 * kb(H), kb(K1)) + packed(2 * kb(H), kb(H)) + packed(N3 / 16, kb(H));
  }

  template<int R>
  int apply_cells(const double *v, double *z, hipStream_t s)
  {
    const int kb1 = kb(K1), kbh = kb(H);
    const size_t lds = 16 * R * (sizeof(float) + sizeof(unsigned short) *
                                                     size_t(32 * (std::max(kb1, kbh) + kbh) + 16));
    if (lds > 64 * 1024)
      AKM_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(mlp_apply_bf16<R>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(lds)));
    const unsigned short *w1 = wbf.data(), *w2 = w1 + packed(2 * kbh, kb1),
                         *w3 = w2 + packed(2 * kbh, kbh);
    const float *p = params.data();
    mlp_apply_bf16<R><<<static_cast<unsigned>((cells + 16 * R - 1) / (16 * R)), 64 * ma_waves, lds,
                        s>>>(cells, N, d, H, N3, kb1, kbh, v, z, feat.data(), w1, p + ob1, w2,
                             p + ob2, w3, p + ob3);
    return check_launch("mlp preconditioner");
  }

  int apply(const double *v, double *z, hipStream_t s) override
  {
    AKM_TRY(refresh_bf16(s));
    // Cells a workgroup: as many as share one reading of the weights while
    // the chip stays full.  16 / 32 / 64 cells took, 256 wide, 64 values:
    // 7.9 / 8.4 / 9.5 us for 4 K cells, 12.4 / 11.6 / 11.1 for 8 K,
    // 23.2 / 16.2 / 15.3 for 16 K and 56 / 41 / 35 for 47 K.
    if (cells <= 16 * 256)
      return apply_cells<1>(v, z, s);
    if (cells <= 32 * 512)
      return apply_cells<2>(v, z, s);
    return apply_cells<4>(v, z, s);
  }
};

static akm_mlp_s *as_mlp(akm_precond p) { return dynamic_cast<akm_mlp_s *>(p); }

extern "C" {

akm_status akm_mlp_create(int d, int n, int64_t num_cells, const int *table, int max_level,
                          int hidden, uint64_t seed, akm_precond *out)
{
  if (out == nullptr || table == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  *out = nullptr;
  if (d < 1 || d > 6 || n < 1 || num_cells < 1 || max_level < 0 || max_level > 30)
    return set_error(AKM_ERR_INVALID, "mlp: invalid grid (d %d, n %d, cells %lld, level %d)", d,
                     n, static_cast<long long>(num_cells), max_level);
  if (hidden <= 0)
    hidden = 256;
  if (hidden % 16 != 0 || hidden > 512)
    return set_error(AKM_ERR_INVALID, "mlp: hidden width %d must be a multiple of 16, <= 512",
                     hidden);
  int64_t N = 1;
  for (int k = 0; k < d; k++)
    N *= n;
  if (N > 256)
    return set_error(AKM_ERR_UNSUPPORTED, "mlp: n^d = %lld above 256", static_cast<long long>(N));
  auto m = std::make_unique<akm_mlp_s>();
  m->d = d;
  m->n = n;
  m->N = static_cast<int>(N);
  m->N3 = static_cast<int>(round16(N));
  m->K1 = static_cast<int>(round16(N + d));
  m->H = hidden;
  m->cells = num_cells;
  m->max_level = max_level;
  const int64_t K1 = m->K1, H = m->H, N3 = m->N3;
  m->oW1 = 0;
  m->ob1 = H * K1;
  m->oW2 = m->ob1 + H;
  m->ob2 = m->oW2 + H * H;
  m->oW3 = m->ob2 + H;
  m->ob3 = m->oW3 + N3 * H;
  m->num_params = m->ob3 + N3;
  // He-normal hidden layers, zero biases, zero output layer (identity map)
  std::vector<float> p(m->num_params, 0.0f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<float> nd(0.0f, 1.0f);
  const float s1 = std::sqrt(2.0f / float(m->N + d)), s2 = std::sqrt(2.0f / float(H));
  for (int64_t j = 0; j < H; j++)
    for (int64_t i = 0; i < m->N + d; i++)
      p[m->oW1 + j * K1 + i] = s1 * nd(rng);
  for (int64_t j = 0; j < H * H; j++)
    p[m->oW2 + j] = s2 * nd(rng);
  AKM_TRY(m->params.upload(p.data(), m->num_params));
  std::vector<float> zeros(m->num_params, 0.0f);
  AKM_TRY(m->adam_m.upload(zeros.data(), m->num_params));
  AKM_TRY(m->adam_v.upload(zeros.data(), m->num_params));
  AKM_TRY(m->grad.upload(zeros.data(), m->num_params));
  AKM_TRY(m->wbf.allocate(m->packed_weights()));
  // features: (level + (position + 1/2) / cells of the level) / (max_level + 1)
  std::vector<float> f(num_cells * d);
  for (int64_t c = 0; c < num_cells; c++)
    for (int k = 0; k < d; k++)
    {
      const int l = table[c * 2 * d + k], pos = table[c * 2 * d + d + k];
      const double count = (l <= 1) ? 1.0 : double(int64_t(1) << (l - 1));
      f[c * d + k] = static_cast<float>((l + (pos + 0.5) / count) / double(max_level + 1));
    }
  AKM_TRY(m->feat.upload(f.data(), num_cells * d));
  *out = m.release();
  return AKM_SUCCESS;
}

akm_status akm_mlp_info(akm_precond p, int64_t *num_params, int *inputs, int *padded_inputs,
                        int *hidden, int *outputs, int *padded_outputs)
{
  auto *m = as_mlp(p);
  if (m == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: not an MLP preconditioner");
  if (num_params)
    *num_params = m->num_params;
  if (inputs)
    *inputs = m->N + m->d;
  if (padded_inputs)
    *padded_inputs = m->K1;
  if (hidden)
    *hidden = m->H;
  if (outputs)
    *outputs = m->N;
  if (padded_outputs)
    *padded_outputs = m->N3;
  return AKM_SUCCESS;
}

akm_status akm_mlp_set_stream(akm_precond p, void *stream)
{
  auto *m = as_mlp(p);
  if (m == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: not an MLP preconditioner");
  m->stream = static_cast<hipStream_t>(stream);
  return AKM_SUCCESS;
}

akm_status akm_mlp_get_params(akm_precond p, float *host)
{
  auto *m = as_mlp(p);
  if (m == nullptr || host == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  AKM_HIP(hipMemcpyAsync(host, m->params.data(), sizeof(float) * m->num_params,
                         hipMemcpyDeviceToHost, m->stream));
  AKM_HIP(hipStreamSynchronize(m->stream));
  return AKM_SUCCESS;
}

akm_status akm_mlp_set_params(akm_precond p, const float *host)
{
  auto *m = as_mlp(p);
  if (m == nullptr || host == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  AKM_HIP(hipMemcpyAsync(m->params.data(), host, sizeof(float) * m->num_params,
                         hipMemcpyHostToDevice, m->stream));
  AKM_HIP(hipStreamSynchronize(m->stream));
  m->bf16_current = false;
  return AKM_SUCCESS;
}

akm_status akm_mlp_forward(akm_precond p, const float *X, int64_t rows, float *O)
{
  auto *m = as_mlp(p);
  if (m == nullptr || X == nullptr || O == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  if (rows < 1 || rows > (1 << 24))
    return set_error(AKM_ERR_INVALID, "mlp: rows %lld out of range", static_cast<long long>(rows));
  AKM_TRY(m->ensure_batch(static_cast<int>(rows)));
  AKM_TRY(m->forward(m->stream, static_cast<int>(rows), X, O));
  AKM_HIP(hipStreamSynchronize(m->stream));
  return AKM_SUCCESS;
}

akm_status akm_mlp_gradients(akm_precond p, const float *X, const float *T, int64_t rows,
                             double *loss, float *grad)
{
  auto *m = as_mlp(p);
  if (m == nullptr || X == nullptr || T == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  if (rows < 1 || rows > (1 << 24))
    return set_error(AKM_ERR_INVALID, "mlp: rows %lld out of range", static_cast<long long>(rows));
  const int B = static_cast<int>(rows);
  AKM_TRY(m->ensure_batch(B));
  AKM_TRY(m->gradients(m->stream, B, X, T, 0, grad != nullptr ? grad : m->grad.data()));
  AKM_HIP(hipStreamSynchronize(m->stream));
  if (loss)
    *loss = *m->host_loss / (double(B) * m->N);
  return AKM_SUCCESS;
}

akm_status akm_mlp_adam_step(akm_precond p, const float *grad, double lr)
{
  auto *m = as_mlp(p);
  if (m == nullptr || grad == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  AKM_TRY(m->adam(m->stream, grad, static_cast<float>(lr)));
  AKM_HIP(hipStreamSynchronize(m->stream));
  return AKM_SUCCESS;
}

akm_status akm_mlp_train(akm_precond p, const double *residuals, const double *corrections,
                         int64_t num_vectors, int epochs, int batch, double lr, uint64_t seed,
                         double *final_loss)
{
  auto *m = as_mlp(p);
  if (m == nullptr || residuals == nullptr || corrections == nullptr)
    return set_error(AKM_ERR_INVALID, "mlp: null argument");
  if (num_vectors < 1 || epochs < 1 || batch < 1 || !(lr > 0))
    return set_error(AKM_ERR_INVALID, "mlp train: vectors %lld, epochs %d, batch %d, lr %g",
                     static_cast<long long>(num_vectors), epochs, batch, lr);
  hipStream_t s = m->stream;
  const int64_t S = num_vectors * m->cells;
  const int B = static_cast<int>(std::min<int64_t>(batch, S));
  AKM_TRY(m->ensure_batch(B));
  dev_buffer<float> X, T;
  dev_buffer<int64_t> perm_d;
  AKM_TRY(X.allocate(S * m->K1));
  AKM_TRY(T.allocate(S * m->N3));
  AKM_TRY(perm_d.allocate(S));
  mlp_make_samples<<<grid_for(S), 256, 0, s>>>(num_vectors, m->cells, m->N, m->d, m->K1, m->N3,
                                               residuals, corrections, m->feat.data(), X.data(),
                                               T.data());
  AKM_TRY(check_launch("mlp samples"));
  std::vector<int64_t> perm(S);
  std::iota(perm.begin(), perm.end(), int64_t{0});
  std::mt19937_64 rng(seed);
  const int64_t nb = S / B; // full batches only
  double epoch_loss = 0;
  for (int ep = 0; ep < epochs; ep++)
  {
    std::shuffle(perm.begin(), perm.end(), rng);
    AKM_HIP(hipMemcpyAsync(perm_d.data(), perm.data(), sizeof(int64_t) * S,
                           hipMemcpyHostToDevice, s));
    for (int64_t bi = 0; bi < nb; bi++)
    {
      mlp_gather<<<B, 256, 0, s>>>(B, perm_d.data(), bi * B, m->K1, m->N3, X.data(), T.data(),
                                    m->Xb.data(), m->Tb.data());
      AKM_TRY(check_launch("mlp gather"));
      AKM_TRY(m->gradients(s, B, m->Xb.data(), m->Tb.data(), bi > 0, m->grad.data()));
      AKM_TRY(m->adam(s, m->grad.data(), static_cast<float>(lr)));
    }
    // the host copy of perm is reshuffled next epoch: wait for the upload
    AKM_HIP(hipStreamSynchronize(s));
    if (ep == epochs - 1)
    {
      double l = 0;
      AKM_HIP(hipMemcpy(&l, m->loss.data(), sizeof(double), hipMemcpyDeviceToHost));
      epoch_loss = l / (double(nb) * B * m->N);
    }
  }
  AKM_TRY(m->refresh_bf16(s));
  AKM_HIP(hipStreamSynchronize(s));
  if (final_loss)
    *final_loss = epoch_loss;
  return AKM_SUCCESS;
}

akm_status akm_precond_apply(akm_precond p, const double *v, double *z, void *stream)
{
  if (p == nullptr || v == nullptr || z == nullptr)
    return set_error(AKM_ERR_INVALID, "precond: null argument");
  return p->apply(v, z, static_cast<hipStream_t>(stream));
}

akm_status akm_precond_destroy(akm_precond p)
{
  delete p;
  return AKM_SUCCESS;
}

} // extern "C"
