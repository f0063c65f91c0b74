// Learned factorized sparse approximate inverse (FSAI) for the lattice Q1 path.
//
// Gridap has no iterative solver (src/Algebra/LinearSolvers.jl:249-303 ships LU
// only); this is the preconditioner of the engine's PCG.  G is lower triangular
// on the pattern of tril(A) and M = GᵀG.  With D = diag(A),
//     G = Ĝ D^(-1/2),   Ĝ_ij = Σ_{cells c ∋ i,j} y_c[pair(i,j)]  (i > j),
//     Ĝ_ii = exp(Σ_{cells c ∋ i} y_c[i]) > 0,
// where y_c (36 numbers: 8 diagonal log-terms, 28 strictly-lower pairs in local
// numbering) is the output of a per-cell MLP 10 -> 64 -> 64 -> 64 -> 36 with GELU,
// BF16 weights and FP32 accumulation.  M is SPD by construction; y = 0 gives
// Ĝ = I, i.e. Jacobi.  Inputs per cell: the cell's share κ_c K̂_aa / A_ii of each of
// its 8 nodes' diagonal (0 at Dirichlet nodes), log κ_c and log h.
//
// Training minimises the probe estimate of ‖I - G A Gᵀ‖²_F / N: for Rademacher z,
// r = z - G A Gᵀ z, L = ‖r‖² / (m N), and on the pattern
//     ∂L/∂G_ij = -2 (r_i v_j + z_i q_j) / (m N),  v = A Gᵀ z,  q = A Gᵀ r,
// then ∂L/∂Ĝ_ij = ∂L/∂G_ij D_jj^(-1/2), gathered to the cells and back-propagated
// through the network.  Every kernel here is deterministic (no float atomics).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "gh_internal.h"

namespace gh {
namespace {

constexpr int kBlock = 256;
constexpr int kEllSlots = kFsaiEllSlots;

inline unsigned grid_for(int64_t n, int block = kBlock) {
  return (unsigned)std::max<int64_t>(1, (n + block - 1) / block);
}

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
  return __uint_as_float((uint32_t)h << 16);
}

// Round to nearest even (finite inputs).
__host__ __device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float gelu(float x) {
  return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}
__device__ __forceinline__ float gelu_d(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) +
         x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// splitmix64 of (seed, probe, index): the Rademacher probe sign.
__host__ __device__ __forceinline__ double rademacher(uint64_t seed, uint64_t probe,
                                                      uint64_t i) {
  uint64_t x = seed + 0x9E3779B97F4A7C15ull * (probe * 0x100000001ull + i + 1ull);
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  x ^= x >> 31;
  return (x & 1ull) ? 1.0 : -1.0;
}

struct Lat3 {
  int nn[3], nc[3];
  double inv0, inv1;
};

__device__ __forceinline__ void node_xyz(const Lat3 &L, int n, int *xi) {
  xi[0] = n % L.nn[0];
  const int t = n / L.nn[0];
  xi[1] = t % L.nn[1];
  xi[2] = t / L.nn[1];
}

// ---- set-up --------------------------------------------------------------

// Per free node: the position and value of its diagonal entry (the number of free
// stencil neighbours below it, from the mask, past the column start) and D^-1/2.
__global__ void diag_setup_kernel(int nnodes, const int32_t *__restrict__ node_dof,
                                  const uint32_t *__restrict__ fmask,
                                  const int32_t *__restrict__ cp, const double *__restrict__ val,
                                  int32_t *__restrict__ dpos, double *__restrict__ diag,
                                  double *__restrict__ fs) {
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  if (node >= nnodes) return;
  const int d = node_dof[node];
  if (d <= 0) return;
  const int p = cp[d - 1] + __popc(fmask[node] & ((1u << 13) - 1u));
  const double v = val[p];
  dpos[d - 1] = p;
  diag[d - 1] = v;
  fs[d - 1] = v > 0.0 ? 1.0 / sqrt(v) : 1.0;
}

__global__ void grf_kappa_kernel(Lat3 L, int64_t ncells, double ox, double oy, double oz,
                                 double hx, double hy, double hz, int nmodes,
                                 const double *__restrict__ omega,
                                 const double *__restrict__ phase, double amp,
                                 double *__restrict__ kappa) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  const int cx = (int)(c % L.nc[0]);
  const int cy = (int)((c / L.nc[0]) % L.nc[1]);
  const int cz = (int)(c / ((int64_t)L.nc[0] * L.nc[1]));
  const double x = ox + (cx + 0.5) * hx, y = oy + (cy + 0.5) * hy, z = oz + (cz + 0.5) * hz;
  double g = 0.0;
  for (int k = 0; k < nmodes; ++k)
    g += cos(omega[3 * k] * x + omega[3 * k + 1] * y + omega[3 * k + 2] * z + phase[k]);
  kappa[c] = exp(amp * g);
}

// ---- network inputs --------------------------------------------------------

// The diagonal comes from its own array, the 8 nodes' loads together: through positions into
// nzval, one node after the other, 62 µs at 64³; now 11 µs.
__global__ void features_kernel(Lat3 L, int64_t ncells, const double *__restrict__ kappa,
                                const int32_t *__restrict__ node_dof,
                                const double *__restrict__ diag, double kdiag, float logh,
                                float *__restrict__ feat) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells) return;
  const int ci = (int)c;
  const int cx = ci % L.nc[0];
  const int cy = (ci / L.nc[0]) % L.nc[1];
  const int cz = ci / (L.nc[0] * L.nc[1]);
  const double k = kappa ? kappa[c] : 1.0;
  int d[8];
  double dg[8];
#pragma unroll
  for (int a = 0; a < 8; ++a)
    d[a] = node_dof[(cx + (a & 1)) + L.nn[0] * ((cy + ((a >> 1) & 1)) + L.nn[1] * (cz + (a >> 2)))];
#pragma unroll
  for (int a = 0; a < 8; ++a) dg[a] = diag[max(d[a], 1) - 1];  // all in flight
  float f[kMlpInPad] = {};
#pragma unroll
  for (int a = 0; a < 8; ++a) f[a] = d[a] > 0 ? (float)(k * kdiag / dg[a]) : 0.0f;
  f[8] = (float)log(k);
  f[9] = logh;
  float4 *out = reinterpret_cast<float4 *>(feat + c * kMlpInPad);
#pragma unroll
  for (int q = 0; q < kMlpInPad / 4; ++q)
    out[q] = make_float4(f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]);
}

// ---- MLP ---------------------------------------------------------------------------

// Inference forward of the whole network on the matrix cores
// (v_mfma_f32_16x16x32_bf16): a wave owns 16-cell tiles; layer inputs are rounded
// to BF16 (A operand: lane l holds cell l%16, inputs 8(l/16)..+7), weights are the
// BF16 values (B operand: output unit l%16, inputs 8(l/16)..+7, kept in registers),
// accumulation is FP32 (D: output unit l%16, cells 4(l/16)..+3).  Bias + GELU are
// applied in FP32 and the activations go through LDS to the next layer's A layout.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kFwdWaves = 4;

__device__ __forceinline__ __bf16 to_bf(float f) {
  const uint16_t h = f32_to_bf16(f);
  __bf16 b;
  memcpy(&b, &h, 2);
  return b;
}
__device__ __forceinline__ __bf16 bf_bits(uint16_t h) {
  __bf16 b;
  memcpy(&b, &h, 2);
  return b;
}

__global__ __launch_bounds__(kFwdWaves * 64) void mlp_fwd_mfma(const float *__restrict__ feat,
                                                               const uint16_t *__restrict__ wq,
                                                               int C, float *__restrict__ yo) {
  __shared__ float act[kFwdWaves][16][kMlpHidden + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const __bf16 zero = to_bf(0.0f);
  v8bf w1[4], w2[4][2], w3[4][2], w4[3][2];
  float b1[4], b2[4], b3[4], b4[3];
  // 8 consecutive BF16 of a 64-wide weight row: one 16-byte load (row offsets are
  // multiples of 8 elements)
  auto row8 = [&](int off) {
    const uint4 u = *reinterpret_cast<const uint4 *>(wq + off);
    v8bf v;
    const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf_bits((uint16_t)(d[i] & 0xffffu));
      v[2 * i + 1] = bf_bits((uint16_t)(d[i] >> 16));
    }
    return v;
  };
  static_assert(kMlpW2 % 8 == 0 && kMlpW3 % 8 == 0 && kMlpW4 % 8 == 0, "aligned rows");
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int n = t * 16 + r16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = kg * 8 + i;
      w1[t][i] = k < kMlpIn ? bf_bits(wq[kMlpW1 + n * kMlpIn + k]) : zero;
    }
#pragma unroll
    for (int sk = 0; sk < 2; ++sk) {
      const int kk = sk * 32 + kg * 8;
      w2[t][sk] = row8(kMlpW2 + n * kMlpHidden + kk);
      w3[t][sk] = row8(kMlpW3 + n * kMlpHidden + kk);
      if (t < 3) {
        if (n < kMlpOut) {
          w4[t][sk] = row8(kMlpW4 + n * kMlpHidden + kk);
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) w4[t][sk][i] = zero;
        }
      }
    }
    b1[t] = bf16_to_f32(wq[kMlpB1 + n]);
    b2[t] = bf16_to_f32(wq[kMlpB2 + n]);
    b3[t] = bf16_to_f32(wq[kMlpB3 + n]);
    if (t < 3) b4[t] = n < kMlpOut ? bf16_to_f32(wq[kMlpB4 + n]) : 0.0f;
  }
  const int ntiles = (C + 15) / 16;
  for (int t0 = blockIdx.x * kFwdWaves; t0 < ntiles; t0 += gridDim.x * kFwdWaves) {
    const int tile = t0 + w;
    const int cell = tile * 16 + r16;
    const bool valid = tile < ntiles && cell < C;
    v8bf a;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = kg * 8 + i;
      a[i] = (valid && k < kMlpInPad) ? to_bf(feat[(size_t)cell * kMlpInPad + k]) : zero;
    }
    v4f acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w1[t], acc[t], 0, 0, 0);
    }
    // hidden layers 2 and 3
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
      const float *bias = layer == 0 ? b1 : b2;
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) act[w][kg * 4 + j][t * 16 + r16] = gelu(acc[t][j] + bias[t]);
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int sk = 0; sk < 2; ++sk) {
        v8bf x;
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = to_bf(act[w][r16][sk * 32 + kg * 8 + i]);
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, layer == 0 ? w2[t][sk] : w3[t][sk],
                                                          acc[t], 0, 0, 0);
      }
    }
    // output layer
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) act[w][kg * 4 + j][t * 16 + r16] = gelu(acc[t][j] + b3[t]);
    __syncthreads();
    v4f out[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) out[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int sk = 0; sk < 2; ++sk) {
      v8bf x;
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = to_bf(act[w][r16][sk * 32 + kg * 8 + i]);
#pragma unroll
      for (int t = 0; t < 3; ++t)
        out[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w4[t][sk], out[t], 0, 0, 0);
    }
    // output-major store yo[n][cell] through LDS: 16 consecutive cells per row
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) act[w][kg * 4 + j][t * 16 + r16] = out[t][j] + b4[t];
    __syncthreads();
    if (tile < ntiles) {
      const int c = tile * 16 + r16;
#pragma unroll
      for (int nb = 0; nb < kMlpOut; nb += 4) {
        const int n = nb + kg;
        if (n < kMlpOut && c < C) yo[(size_t)n * C + c] = act[w][r16][n];
      }
    }
  }
}

// Training: forward, and forward + backward, on the FP32 matrix cores
// (v_mfma_f32_16x16x4_f32: FP32 operands and accumulators; lane l supplies A[l%16][k],
// B[k][l%16] with k of its lane group l/16, and holds D[4(l/16)+j][l%16]).  A workgroup
// takes tiles of 64 cells; a wave owns 16 of them in the forward and the
// back-propagated products (cells are the rows, the layer's units the columns) and 16
// output units in the weight gradients (units are the rows, the 64 cells the
// contraction).  The order of a contraction is free, so group g takes k = 16 g + kk: each
// lane's 16 operands are contiguous, in LDS and in the BF16 weights (read from L1).
// The backward kernel recomputes the activations from the features: it reads 64 B
// of features and 160 B of output gradient per cell and keeps the rest in LDS, and each
// workgroup writes one partial of every gradient; an FP32 sum covers at most 256 cells
// however large the mesh (kRunTiles).  Bound by the matrix cores at large
// C (560 instructions of 32 cycles per tile and wave), by the number of tiles below
// 256 tiles.  One lane per unit and 256 cells in turn left 128 waves for the whole chip:
// 32³ cells 1,480 µs for forward, backward, gradients and their sums; now 20 + 58 + 9 µs.
constexpr int kTrainCells = 64;
constexpr int kTrainLd = kMlpHidden + 4;   // row stride of activations: conflict-free b128
constexpr int kTrainGrid = 256;            // most workgroups of the backward (partials)
constexpr int kRunTiles = 4;               // most tiles that one FP32 gradient sum covers

struct TrainLds {
  float h[3][kTrainCells][kTrainLd];   // activations, then (backward) pre-activation gradients
  float dy[kTrainCells][48 + 4];       // output gradient, zero from 36 on
  float ft[kTrainCells][kMlpInPad + 4];  // features; column 10 is 1 (the bias gradient)
};

__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int N>
__device__ __forceinline__ void load_row(const float *p, float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const float4 q = reinterpret_cast<const float4 *>(p)[i];
    v[4 * i] = q.x;
    v[4 * i + 1] = q.y;
    v[4 * i + 2] = q.z;
    v[4 * i + 3] = q.w;
  }
}

// 16 consecutive BF16 weights as FP32 (16-byte aligned)
__device__ __forceinline__ void load_weights16(const uint16_t *w, float (&v)[16]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint4 u = reinterpret_cast<const uint4 *>(w)[i];
    const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[8 * i + 2 * j] = __uint_as_float(d[j] << 16);
      v[8 * i + 2 * j + 1] = __uint_as_float(d[j] & 0xffff0000u);
    }
  }
}

// The three hidden layers of the wave's 16 cells: activations to S.h, gelu' of the
// pre-activations to gd (BWD).
template <bool BWD>
__device__ __forceinline__ void hidden_layers(TrainLds &S, const uint16_t *__restrict__ wq,
                                              int wave, int lane, float (&gd)[3][16]) {
  const int l16 = lane & 15, g = lane >> 4, row = 16 * wave + l16;
#pragma unroll
  for (int layer = 0; layer < 3; ++layer) {
    const int woff = layer == 0 ? kMlpW1 : layer == 1 ? kMlpW2 : kMlpW3;
    const int boff = layer == 0 ? kMlpB1 : layer == 1 ? kMlpB2 : kMlpB3;
    float a[16];
    if (layer == 0) {
      float f[4];
      load_row(&S.ft[row][4 * g], f);
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = f[k];
    } else {
      load_row(&S.h[layer - 1][row][16 * g], a);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int unit = 16 * t + l16;
      v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
      if (layer == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          acc = mfma4(a[k], 4 * g + k < kMlpIn
                                ? bf16_to_f32(wq[kMlpW1 + unit * kMlpIn + 4 * g + k]) : 0.0f, acc);
      } else {
        float w[16];
        load_weights16(wq + woff + unit * kMlpHidden + 16 * g, w);
#pragma unroll
        for (int k = 0; k < 16; ++k) acc = mfma4(a[k], w[k], acc);
      }
      const float bias = bf16_to_f32(wq[boff + unit]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float z = acc[j] + bias;
        S.h[layer][16 * wave + 4 * g + j][unit] = gelu(z);
        if (BWD) gd[layer][4 * t + j] = gelu_d(z);
      }
    }
    wave_sync();  // the wave reads its own 16 rows next
  }
}

// features of a tile to LDS (rows past the last cell are zero)
__device__ __forceinline__ void load_features(TrainLds &S, const float *__restrict__ feat, int c0,
                                              int C) {
  const int r = threadIdx.x >> 2, q = threadIdx.x & 3;  // 64 rows x 4 quads
  float4 v{0.0f, 0.0f, 0.0f, 0.0f};
  if (c0 + r < C) v = reinterpret_cast<const float4 *>(feat + (size_t)(c0 + r) * kMlpInPad)[q];
  if (q == 2) v.z = 1.0f;
  *reinterpret_cast<float4 *>(&S.ft[r][4 * q]) = v;
}

// network output yo[n][cell] of every cell
__global__ __launch_bounds__(256) void mlp_train_fwd(const float *__restrict__ feat,
                                                     const uint16_t *__restrict__ wq, int C,
                                                     float *__restrict__ yo) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  TrainLds &S = *reinterpret_cast<TrainLds *>(lds_raw);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  float gd[3][16];
  for (int c0 = blockIdx.x * kTrainCells; c0 < C; c0 += gridDim.x * kTrainCells) {
    __syncthreads();
    load_features(S, feat, c0, C);
    __syncthreads();
    hidden_layers<false>(S, wq, wave, lane, gd);
    float a[16];
    load_row(&S.h[2][16 * wave + l16][16 * g], a);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const int n = 16 * t + l16;
      float w[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) w[k] = 0.0f;
      if (n < kMlpOut) load_weights16(wq + kMlpW4 + n * kMlpHidden + 16 * g, w);
      v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 16; ++k) acc = mfma4(a[k], w[k], acc);
      if (n < kMlpOut) {
        const float bias = bf16_to_f32(wq[kMlpB4 + n]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int c = c0 + 16 * wave + 4 * g + j;
          if (c < C) yo[(size_t)n * C + c] = acc[j] + bias;
        }
      }
    }
  }
}

// Weights in input-major order (the backward product's B operand), in LDS
constexpr int kWtLd = kMlpHidden + 8;      // BF16; 16-byte rows, conflict-free b128
constexpr int kWt4Ld = 56;                 // 36 outputs padded to 48
struct TrainWeights {
  uint16_t w2t[kMlpHidden][kWtLd], w3t[kMlpHidden][kWtLd], w4t[kMlpHidden][kWt4Ld];
};

// Partial gradients of every weight: one kMlpParams run per workgroup.  LONG, for workgroups
// of more than kRunTiles tiles: every kRunTiles tiles the FP32 sums go to FP64 ones, in
// registers (74 of the 512 of one wave on a SIMD) and, W2's, in LDS (a thread's own; all in
// registers spill).  Step at 64³ and 96³: FP32 throughout 0.768 and 2.452 ms with gradient
// errors of 4e-8 and 6e-8 of the FP64 evaluation, LONG 0.782 and 2.502 ms and 3e-8 at both; a
// partial for every run 0.800 and 2.568 ms, a workgroup for every run 0.815 and 2.664.
template <bool LONG>
__global__ __launch_bounds__(256) void mlp_train_bwd(const float *__restrict__ feat,
                                                     const uint16_t *__restrict__ wq,
                                                     const float *__restrict__ dy, int C,
                                                     float *__restrict__ part) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  TrainLds &S = *reinterpret_cast<TrainLds *>(lds_raw);
  TrainWeights &W = *reinterpret_cast<TrainWeights *>(lds_raw + sizeof(TrainLds));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int row = 16 * wave + l16;
  for (int t = threadIdx.x; t < kMlpHidden * kMlpHidden; t += 256) {
    const int o = t / kMlpHidden, i = t % kMlpHidden;
    W.w2t[i][o] = wq[kMlpW2 + t];
    W.w3t[i][o] = wq[kMlpW3 + t];
    if (o < 48) W.w4t[i][o] = o < kMlpOut ? wq[kMlpW4 + o * kMlpHidden + i] : (uint16_t)0;
  }
  // this wave's gradient tiles: W2, W3 rows 16 wave.. x all inputs; W4 all outputs x inputs
  // 16 wave..; W1 rows 16 wave.. x the (padded) inputs
  v4f aw1{0.0f, 0.0f, 0.0f, 0.0f}, aw2[4], aw3[4], aw4[3];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    aw2[t] = aw3[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if (t < 3) aw4[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  }
  float ab2 = 0.0f, ab3 = 0.0f, ab4[3] = {0.0f, 0.0f, 0.0f};
  // LONG: the same in FP64 over the runs so far (entry e of W2's at sw2[256 e])
  double sw1[4] = {}, sw3[4][4] = {}, sw4[3][4] = {}, sb2 = 0.0, sb3 = 0.0, sb4[3] = {};
  double *sw2 = reinterpret_cast<double *>(lds_raw + sizeof(TrainLds) + sizeof(TrainWeights)) +
                threadIdx.x;
  if (LONG)
#pragma unroll
    for (int e = 0; e < 16; ++e) sw2[256 * e] = 0.0;
  auto end_run = [&] {
    auto move = [](float a, double &s) { s += (double)a; };
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      move(aw1[j], sw1[j]);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        move(aw2[t][j], sw2[256 * (4 * t + j)]);
        move(aw3[t][j], sw3[t][j]);
        if (t < 3) move(aw4[t][j], sw4[t][j]);
      }
    }
    move(ab2, sb2);
    move(ab3, sb3);
    aw1 = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    ab2 = ab3 = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      aw2[t] = aw3[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      if (t < 3) {
        aw4[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        move(ab4[t], sb4[t]);
        ab4[t] = 0.0f;
      }
    }
  };
  int tiles = 0;
  float gd[3][16];
  // contraction step s of a weight gradient: the cell of lane group g (rows four apart,
  // so the groups of a half-wave read different banks)
  auto cell_of = [&](int s) { return 4 * g + (s & 3) + 16 * (s >> 2); };
  // pre-activation gradient of a hidden layer: rows a (the layer above's gradient), its
  // weights input-major, times gelu'; written over the activations
  auto back16 = [&](int from, int to, const uint16_t (*wt)[kWtLd]) {
    float a[16], d[16];
    load_row(&S.h[from][row][16 * g], a);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float w[16];
      load_weights16(&wt[16 * t + l16][16 * g], w);
      v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 16; ++k) acc = mfma4(a[k], w[k], acc);
#pragma unroll
      for (int j = 0; j < 4; ++j) d[4 * t + j] = acc[j] * gd[to][4 * t + j];
    }
    __syncthreads();  // every wave has read the activations
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) S.h[to][16 * wave + 4 * g + j][16 * t + l16] = d[4 * t + j];
    __syncthreads();
  };
  for (int c0 = blockIdx.x * kTrainCells; c0 < C; c0 += gridDim.x * kTrainCells) {
    __syncthreads();
    load_features(S, feat, c0, C);
    for (int t = threadIdx.x; t < kTrainCells * 12; t += 256) {  // 12 quads, 9 of them stored
      const int r = t / 12, q = t % 12;
      float4 v{0.0f, 0.0f, 0.0f, 0.0f};
      if (c0 + r < C && q < kMlpOut / 4)
        v = reinterpret_cast<const float4 *>(dy + (size_t)(c0 + r) * kMlpOutPad)[q];
      *reinterpret_cast<float4 *>(&S.dy[r][4 * q]) = v;
    }
    __syncthreads();
    hidden_layers<true>(S, wq, wave, lane, gd);
    __syncthreads();
    // output layer: dW4 = dyᵀ h3, db4, and dz3
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int c = cell_of(s);
      const float b = S.h[2][c][16 * wave + l16];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const float a = S.dy[c][16 * t + l16];
        aw4[t] = mfma4(a, b, aw4[t]);
        ab4[t] += a;
      }
    }
    {
      float a[12], d[16];
      load_row(&S.dy[row][12 * g], a);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint2 *wp = reinterpret_cast<const uint2 *>(&W.w4t[16 * t + l16][12 * g]);
        v4f acc{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const uint2 u = wp[q];
          acc = mfma4(a[4 * q], __uint_as_float(u.x << 16), acc);
          acc = mfma4(a[4 * q + 1], __uint_as_float(u.x & 0xffff0000u), acc);
          acc = mfma4(a[4 * q + 2], __uint_as_float(u.y << 16), acc);
          acc = mfma4(a[4 * q + 3], __uint_as_float(u.y & 0xffff0000u), acc);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) d[4 * t + j] = acc[j] * gd[2][4 * t + j];
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) S.h[2][16 * wave + 4 * g + j][16 * t + l16] = d[4 * t + j];
      __syncthreads();
    }
    // hidden layer 3: dW3 = dz3ᵀ h2; hidden layer 2: dW2 = dz2ᵀ h1
    auto wgrad = [&](int layer, v4f (&aw)[4], float &ab) {
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        const int c = cell_of(s);
        const float a = S.h[layer][c][16 * wave + l16];
        ab += a;
#pragma unroll
        for (int t = 0; t < 4; ++t) aw[t] = mfma4(a, S.h[layer - 1][c][16 * t + l16], aw[t]);
      }
    };
    wgrad(2, aw3, ab3);
    back16(2, 1, W.w3t);
    wgrad(1, aw2, ab2);
    back16(1, 0, W.w2t);
    // input layer: dW1 = dz1ᵀ features (column 10 of the features is 1: db1)
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const int c = cell_of(s);
      aw1 = mfma4(S.h[0][c][16 * wave + l16], S.ft[c][l16], aw1);
    }
    if (LONG && ++tiles % kRunTiles == 0) end_run();
  }
  // bias sums over the lane groups
  auto groups = [](auto v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
  if constexpr (LONG) {
    end_run();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      aw1[j] = (float)sw1[j];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        aw2[t][j] = (float)sw2[256 * (4 * t + j)];
        aw3[t][j] = (float)sw3[t][j];
        if (t < 3) aw4[t][j] = (float)sw4[t][j];
      }
    }
    ab2 = (float)groups(sb2);
    ab3 = (float)groups(sb3);
#pragma unroll
    for (int t = 0; t < 3; ++t) ab4[t] = (float)groups(sb4[t]);
  } else {
    ab2 = groups(ab2);
    ab3 = groups(ab3);
#pragma unroll
    for (int t = 0; t < 3; ++t) ab4[t] = groups(ab4[t]);
  }
  float *pp = part + (size_t)blockIdx.x * kMlpParams;
  if (g == 0) {
    pp[kMlpB2 + 16 * wave + l16] = ab2;
    pp[kMlpB3 + 16 * wave + l16] = ab3;
    if (wave == 0)
#pragma unroll
      for (int t = 0; t < 3; ++t)
        if (16 * t + l16 < kMlpOut) pp[kMlpB4 + 16 * t + l16] = ab4[t];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int o = 16 * wave + 4 * g + j;
    if (l16 < kMlpIn) pp[kMlpW1 + o * kMlpIn + l16] = aw1[j];
    else if (l16 == kMlpIn) pp[kMlpB1 + o] = aw1[j];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      pp[kMlpW2 + o * kMlpHidden + 16 * t + l16] = aw2[t][j];
      pp[kMlpW3 + o * kMlpHidden + 16 * t + l16] = aw3[t][j];
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const int n = 16 * t + 4 * g + j;
      if (n < kMlpOut) pp[kMlpW4 + n * kMlpHidden + 16 * wave + l16] = aw4[t][j];
    }
  }
}

// Gradient of every parameter: its partials summed in FP64 in a fixed order (16 threads
// a parameter), then the Adam step (lr > 0).
constexpr int kReduceLanes = 16;
__global__ __launch_bounds__(256) void reduce_adam_kernel(
    const float *__restrict__ part, int nblocks, float *__restrict__ g, float lr, float b1t,
    float b2t, float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
    uint16_t *__restrict__ wq) {
  constexpr int P = 256 / kReduceLanes;  // parameters per workgroup: 64-byte runs of a partial
  __shared__ double sh[kReduceLanes][P];
  const int col = threadIdx.x % P, lane = threadIdx.x / P;
  const int t = blockIdx.x * P + col;
  double s = 0.0;
  if (t < kMlpParams) {
    constexpr int U = kTrainGrid / kReduceLanes;  // partials per thread, all in flight
    float x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int b = lane + u * kReduceLanes;
      x[u] = b < nblocks ? part[(size_t)b * kMlpParams + t] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s += x[u];
  }
  sh[lane][col] = s;
  __syncthreads();
  if (lane != 0 || t >= kMlpParams) return;
  s = 0.0;
#pragma unroll
  for (int k = 0; k < kReduceLanes; ++k) s += sh[k][col];
  const float gi = (float)s;
  g[t] = gi;
  if (!(lr > 0.0f)) return;
  const float mi = 0.9f * m[t] + 0.1f * gi;
  const float vi = 0.999f * v[t] + 0.001f * gi * gi;
  m[t] = mi;
  v[t] = vi;
  const float wi = w[t] - lr * (mi / (1.0f - b1t)) / (sqrtf(vi / (1.0f - b2t)) + 1e-8f);
  w[t] = wi;
  wq[t] = f32_to_bf16(wi);
}

__global__ void to_bf16_kernel(int n, const float *__restrict__ w, uint16_t *__restrict__ wq) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) wq[t] = f32_to_bf16(w[t]);
}

// ---- Ĝ from the cell outputs (owner computes: one thread per lattice node) ----

__device__ __forceinline__ int pair_index(int a, int b) {  // a > b, local numbering
  return 8 + a * (a - 1) / 2 + b;
}

// One thread per lattice node n (row i of G).  The entry of n and its neighbour at offset
// o is Σ over the cells holding both, in ascending cell order (both endpoints compute the
// same bits); n is local node 7 ^ e of its e-th cell, so its 8 cells give 8 values each:
// 64 loads, all in flight (cells outside the lattice read cell 0 and count 0).  Summed
// inside a branch per neighbour and cell, as before, every load waited for the one
// before (64³: 75 µs, now 51; 32³ with the CSC copies 36 µs, now 8).
// Written: the column-i prefix (gl, rows of G) and suffix (gu, rows of Gᵀ) of Ĝ in CSC
// positions (CSC), and (solver) the solver's copy of G = Ĝ D^-1/2 in 16-slot rows:
// gle[i] = G(i, j ≤ i), gue[i] = G(j ≥ i, i).
template <bool CSC>
__global__ __launch_bounds__(64) void g_assemble_kernel(
    Lat3 L, int nnodes, const int32_t *__restrict__ node_dof, const uint32_t *__restrict__ fmask,
    const int32_t *__restrict__ colptr, const float *__restrict__ yo,
    const double *__restrict__ fs, float *__restrict__ gl, float *__restrict__ gu, bool solver,
    float *__restrict__ gle, float *__restrict__ gue, int64_t nfree, float *__restrict__ g14) {
  const int n = blockIdx.x * 64 + threadIdx.x;
  if (n >= nnodes) return;
  const int d0 = node_dof[n];
  if (d0 <= 0) return;
  int xi[3];
  node_xyz(L, n, xi);
  const uint32_t fm = fmask[n];
  const int p0 = colptr[d0 - 1];
  const int C = L.nc[0] * L.nc[1] * L.nc[2];
  float v[8][8];  // v[e][b]: cell e's value of the pair (n, its local node b)
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int cx = xi[0] - 1 + (e & 1), cy = xi[1] - 1 + ((e >> 1) & 1), cz = xi[2] - 1 + (e >> 2);
    const bool in = cx >= 0 && cx < L.nc[0] && cy >= 0 && cy < L.nc[1] && cz >= 0 && cz < L.nc[2];
    const int cell = in ? cx + L.nc[0] * (cy + L.nc[1] * cz) : 0;
    const int a = 7 ^ e;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int idx = a == b ? a : (a > b ? pair_index(a, b) : pair_index(b, a));
      const float y = yo[(size_t)idx * C + cell];
      v[e][b] = in ? y : 0.0f;
    }
  }
  const double sn = fs[d0 - 1];
  // D^-1/2 of the lower neighbours (the node itself where there is none)
  double sm[13];
  if (solver) {
    int dm[13];
#pragma unroll
    for (int o = 0; o < 13; ++o)
      dm[o] = node_dof[(fm >> o) & 1u ? n + (o % 3 - 1) + L.nn[0] * (((o / 3) % 3 - 1) +
                                                                   L.nn[1] * (o / 9 - 1))
                                      : n];
#pragma unroll
    for (int o = 0; o < 13; ++o) sm[o] = fs[dm[o] - 1];
  }
  float *el = gle + (size_t)(d0 - 1) * kEllSlots, *eu = gue + (size_t)(d0 - 1) * kEllSlots;
  int kl = 0, ku = 0;
#pragma unroll
  for (int o = 0; o < 27; ++o) {
    const int dx = o % 3 - 1, dy = (o / 3) % 3 - 1, dz = o / 9 - 1;
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int a = 7 ^ e;
      const int bx = (a & 1) + dx, by = ((a >> 1) & 1) + dy, bz = (a >> 2) + dz;
      if (bx >= 0 && bx <= 1 && by >= 0 && by <= 1 && bz >= 0 && bz <= 1)
        sum += v[e][bx | (by << 1) | (bz << 2)];
    }
    if (!((fm >> o) & 1u)) {
      // lower offsets whose neighbour is not free (outside the box): zero
      if (o < 13 && solver && g14) g14[o * nfree + (d0 - 1)] = 0.0f;
      continue;
    }
    const int pos = p0 + __popc(fm & ((1u << o) - 1u));
    if (o == 13) {
      const float g = expf(sum);
      if (CSC) {
        gl[pos] = g;
        gu[pos] = g;
      }
      if (solver) {
        const float ge = (float)((double)g * sn);
        el[kl++] = ge;
        eu[ku++] = ge;
        if (g14) g14[13 * nfree + (d0 - 1)] = ge;
      }
    } else if (o < 13) {
      if (CSC) gl[pos] = sum;  // Ĝ(n, m), m < n
      if (solver) {
        const float ge = (float)((double)sum * sm[o]);
        el[kl++] = ge;
        if (g14) g14[o * nfree + (d0 - 1)] = ge;
      }
    } else {
      if (CSC) gu[pos] = sum;  // Ĝ(m, n), m > n
      if (solver) eu[ku++] = (float)((double)sum * sn);
    }
  }
  if (solver) {
    for (; kl < kEllSlots; ++kl) el[kl] = 0.0f;
    for (; ku < kEllSlots; ++ku) eu[ku] = 0.0f;
  }
}

// Column indices of the 16-slot rows (from the pattern; padding points at the row
// itself, with zero weight); flags rows whose halves exceed 16 entries.
__global__ void ell_index_kernel(int64_t n, const int32_t *__restrict__ cp,
                                 const int32_t *__restrict__ rv, const int32_t *__restrict__ dpos,
                                 int32_t *__restrict__ gli, int32_t *__restrict__ gui,
                                 int *__restrict__ overflow) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int lo = cp[i], d = dpos[i], hi = cp[i + 1];
  if (d - lo + 1 > kEllSlots || hi - d > kEllSlots) atomicOr(overflow, 1);
  for (int k = 0; k < kEllSlots; ++k) {
    gli[i * kEllSlots + k] = lo + k <= d ? rv[lo + k] : (int32_t)i;
    gui[i * kEllSlots + k] = d + k < hi ? rv[d + k] : (int32_t)i;
  }
}

// ∂L/∂y_c from the pattern gradient (the transpose of g_assemble).  The 36 gradient
// loads of a cell are independent (a pair with a Dirichlet node reads entry 0 and
// counts 0): 21 -> 7 µs at 32³.
__global__ __launch_bounds__(64) void cell_grad_kernel(
    Lat3 L, int ncells, const int32_t *__restrict__ node_dof, const uint32_t *__restrict__ fmask,
    const int32_t *__restrict__ colptr, const float *__restrict__ gG,
    const float *__restrict__ gl, float *__restrict__ dy) {
  const int c = blockIdx.x * 64 + threadIdx.x;
  if (c >= ncells) return;
  const int cx = c % L.nc[0];
  const int cy = (c / L.nc[0]) % L.nc[1];
  const int cz = c / (L.nc[0] * L.nc[1]);
  int dof[8], cp[8];
  uint32_t fm[8];
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const int node = (cx + (a & 1)) + L.nn[0] * ((cy + ((a >> 1) & 1)) + L.nn[1] * (cz + (a >> 2)));
    dof[a] = node_dof[node];
    fm[a] = fmask[node];
  }
#pragma unroll
  for (int a = 0; a < 8; ++a) cp[a] = colptr[max(dof[a], 1) - 1];
  float out[kMlpOutPad] = {};
  float gd[8];
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const int pd = dof[a] > 0 ? cp[a] + __popc(fm[a] & ((1u << 13) - 1u)) : 0;
    out[a] = gG[pd];
    gd[a] = gl[pd];
  }
#pragma unroll
  for (int a = 1; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < a; ++b) {
      const int o = ((b & 1) - (a & 1) + 1) + 3 * (((b >> 1) & 1) - ((a >> 1) & 1) + 1) +
                    9 * ((b >> 2) - (a >> 2) + 1);
      const bool in = dof[a] > 0 && dof[b] > 0;
      const float g = gG[in ? cp[a] + __popc(fm[a] & ((1u << o) - 1u)) : 0];
      out[pair_index(a, b)] = in ? g : 0.0f;
    }
#pragma unroll
  for (int a = 0; a < 8; ++a) out[a] = dof[a] > 0 ? out[a] * gd[a] : 0.0f;
  float4 *p = reinterpret_cast<float4 *>(dy + (size_t)c * kMlpOutPad);
#pragma unroll
  for (int q = 0; q < kMlpOutPad / 4; ++q)
    p[q] = make_float4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
}

// ---- probes -----------------------------------------------------------------------------
// NB probes at a time, their vectors interleaved ([row][NB]), so that the matrix and the
// factor are read once per batch and a column is one gather of NB values.  A row's
// entries are spread over its lanes, all of a turn's loads in flight (four kernels per
// probe with one entry at a time: 40 µs and 8 launches a probe at 32³; now 31 µs and 7
// launches for four).

constexpr int kApplyLanes = 4, kApplyTurn = 4;   // a half row: at most 14 entries of 16
constexpr int kMultiLanes = 8, kMultiTurn = 4;   // a full row: at most 27 of 32

// bit k of sg[i]: the sign of probe first + k at i (set: +1)
__global__ void rademacher_kernel(int64_t n, uint64_t seed, uint64_t first, int nb,
                                  uint8_t *__restrict__ sg) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t m = 0;
  for (int k = 0; k < nb; ++k)
    m |= (rademacher(seed, first + (uint64_t)k, (uint64_t)i) > 0.0 ? 1u : 0u) << k;
  sg[i] = (uint8_t)m;
}

template <int NB>
struct Vals {
  double v[NB];
};
template <int NB>
__device__ __forceinline__ Vals<NB> signs(const uint8_t *__restrict__ sg, int64_t i) {
  const uint32_t m = sg[i];
  Vals<NB> r;
#pragma unroll
  for (int k = 0; k < NB; ++k) r.v[k] = (m >> k) & 1u ? 1.0 : -1.0;
  return r;
}
template <int NB>
__device__ __forceinline__ Vals<NB> load_vals(const double *__restrict__ x, int64_t i) {
  Vals<NB> r;
  if constexpr (NB % 2 == 0) {
#pragma unroll
    for (int k = 0; k < NB; k += 2) {
      const double2 d = *reinterpret_cast<const double2 *>(x + i * NB + k);
      r.v[k] = d.x;
      r.v[k + 1] = d.y;
    }
  } else {
#pragma unroll
    for (int k = 0; k < NB; ++k) r.v[k] = x[i * NB + k];
  }
  return r;
}

// s_k += Σ over entries [p0, p1) of the row, L lanes and U entries each: wt(p) f(rv[p])
template <int L, int U, int NB, class Wt, class F>
__device__ __forceinline__ void row_dot(int p0, int p1, const int32_t *__restrict__ rv, Wt wt,
                                        F f, double (&s)[NB]) {
  const int sub = threadIdx.x % L;
  for (int p = p0; p < p1; p += L * U) {
    int j[U];
    double w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = min(p + sub + u * L, p1 - 1);
      j[u] = rv[q];
      w[u] = wt(q);
    }
    Vals<NB> g[U];
#pragma unroll
    for (int u = 0; u < U; ++u) g[u] = f(j[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p + sub + u * L < p1)
#pragma unroll
        for (int k = 0; k < NB; ++k) s[k] += w[u] * g[u].v[k];
  }
#pragma unroll
  for (int k = 0; k < NB; ++k)
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) s[k] += __shfl_xor(s[k], o);
}

// z_j = s_j Σ_{i >= j} Ĝ_ij y_i  (column-j suffix); SIGNS: y are the probes themselves
template <int NB, bool SIGNS>
__global__ __launch_bounds__(256) void apply_upper_kernel(
    int64_t n, const int32_t *__restrict__ cp, const int32_t *__restrict__ rv,
    const int32_t *__restrict__ dpos, const float *__restrict__ gu,
    const double *__restrict__ fs, const uint8_t *__restrict__ sg, const double *__restrict__ y,
    double *__restrict__ z) {
  const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kApplyLanes;
  double s[NB] = {};
  if (row < n)
    row_dot<kApplyLanes, kApplyTurn, NB>(
        dpos[row], cp[row + 1], rv, [&](int p) { return (double)gu[p]; },
        [&](int j) {
          if constexpr (SIGNS) return signs<NB>(sg, j);
          else return load_vals<NB>(y, j);
        },
        s);
  if (row < n && threadIdx.x % kApplyLanes == 0) {
    const double f = fs[row];
#pragma unroll
    for (int k = 0; k < NB; ++k) z[row * NB + k] = f * s[k];
  }
}

// y = A x
template <int NB>
__global__ __launch_bounds__(256) void spmv_multi_kernel(
    int64_t n, const int32_t *__restrict__ cp, const int32_t *__restrict__ rv,
    const double *__restrict__ val, const double *__restrict__ x, double *__restrict__ y) {
  const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kMultiLanes;
  double s[NB] = {};
  if (row < n)
    row_dot<kMultiLanes, kMultiTurn, NB>(
        cp[row], cp[row + 1], rv, [&](int p) { return val[p]; },
        [&](int j) { return load_vals<NB>(x, j); }, s);
  if (row < n && threadIdx.x % kMultiLanes == 0)
#pragma unroll
    for (int k = 0; k < NB; ++k) y[row * NB + k] = s[k];
}

// r = z − u, u_i = Σ_{j <= i} Ĝ_ij s_j v_j (column-i prefix); block partials of r·r over
// the probes, added to lpart (one slot per block)
template <int NB>
__global__ __launch_bounds__(256) void residual_kernel(
    int64_t n, const int32_t *__restrict__ cp, const int32_t *__restrict__ rv,
    const int32_t *__restrict__ dpos, const float *__restrict__ gl,
    const double *__restrict__ fs, const uint8_t *__restrict__ sg, const double *__restrict__ v,
    double *__restrict__ r, double *__restrict__ lpart) {
  __shared__ double sh[4];
  double acc = 0.0;
  const int64_t step = (int64_t)gridDim.x * (256 / kApplyLanes);
  for (int64_t r0 = (int64_t)blockIdx.x * (256 / kApplyLanes); r0 < n; r0 += step) {
    const int64_t row = r0 + threadIdx.x / kApplyLanes;
    double s[NB] = {};
    if (row < n)
      row_dot<kApplyLanes, kApplyTurn, NB>(
          cp[row], dpos[row] + 1, rv, [&](int p) { return (double)gl[p]; },
          [&](int j) {
            Vals<NB> x = load_vals<NB>(v, j);
            const double f = fs[j];
#pragma unroll
            for (int k = 0; k < NB; ++k) x.v[k] *= f;
            return x;
          },
          s);
    if (row < n && threadIdx.x % kApplyLanes == 0) {
      const Vals<NB> z = signs<NB>(sg, row);
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const double ri = z.v[k] - s[k];
        r[row * NB + k] = ri;
        acc += ri * ri;
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) lpart[blockIdx.x] += sh[0] + sh[1] + sh[2] + sh[3];
}

// gĜ_ij (+)= coef Σ_k (r_i v_j + z_i q_j) s_j on the lower pattern (column-i prefix); the
// first batch writes
template <int NB>
__global__ __launch_bounds__(256) void pattern_grad_kernel(
    int64_t n, const int32_t *__restrict__ cp, const int32_t *__restrict__ rv,
    const int32_t *__restrict__ dpos, const double *__restrict__ fs,
    const double *__restrict__ r, const double *__restrict__ v, const uint8_t *__restrict__ sg,
    const double *__restrict__ q, double coef, bool add, float *__restrict__ gG) {
  const int64_t row = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kApplyLanes;
  if (row >= n) return;
  const Vals<NB> ri = load_vals<NB>(r, row), zi = signs<NB>(sg, row);
  const int p0 = cp[row] + threadIdx.x % kApplyLanes, p1 = dpos[row];
  for (int p = p0; p <= p1; p += kApplyLanes * kApplyTurn) {
    int j[kApplyTurn];
    double f[kApplyTurn];
    Vals<NB> vj[kApplyTurn], qj[kApplyTurn];
#pragma unroll
    for (int u = 0; u < kApplyTurn; ++u) j[u] = rv[min(p + u * kApplyLanes, p1)];
#pragma unroll
    for (int u = 0; u < kApplyTurn; ++u) {
      vj[u] = load_vals<NB>(v, j[u]);
      qj[u] = load_vals<NB>(q, j[u]);
      f[u] = fs[j[u]];
    }
#pragma unroll
    for (int u = 0; u < kApplyTurn; ++u) {
      const int at = p + u * kApplyLanes;
      if (at > p1) continue;
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < NB; ++k) t += ri.v[k] * vj[u].v[k] + zi.v[k] * qj[u].v[k];
      const float d = (float)(coef * t * f[u]);
      gG[at] = add ? gG[at] + d : d;
    }
  }
}

Lat3 lattice_of(const Ctx &c) {
  Lat3 L;
  for (int k = 0; k < 3; ++k) {
    L.nn[k] = (int)(c.part[k] + 1);
    L.nc[k] = (int)c.part[k];
  }
  L.inv0 = 1.0 / L.nn[0];
  L.inv1 = 1.0 / L.nn[1];
  return L;
}

constexpr int kResidualBlocks = 512;
constexpr int kProbeBatch = 4;

}  // namespace

void fsai_prepare(Ctx &c) {
  GH_REQUIRE(c.structured && c.cartesian && c.dim == 3, GH_ERR_UNSUPPORTED,
             "the learned FSAI needs a 3-D Cartesian mesh with a scalar Q1 CLagrangian space");
  GH_REQUIRE(c.have_values, GH_ERR_STATE, "assemble the matrix before the FSAI set-up");
  const int64_t n = c.nfree, C = c.ncells;
  if (!c.fsai_ready) {
    c.diagpos.resize(std::max<int64_t>(n, 1));
    c.diag.resize(std::max<int64_t>(n, 1));
    c.fs.resize(std::max<int64_t>(n, 1));
    c.gl.resize(std::max<int64_t>(c.nnz, 1));
    c.gu.resize(std::max<int64_t>(c.nnz, 1));
    c.feat.resize(C * kMlpInPad);
    c.yo.resize(C * kMlpOut);  // output-major: yo[n * C + cell]
    for (auto *b : {&c.gle, &c.gue}) b->resize((size_t)std::max<int64_t>(n, 1) * kEllSlots);
    for (auto *b : {&c.gli, &c.gui}) b->resize((size_t)std::max<int64_t>(n, 1) * kEllSlots);
  }
  hipLaunchKernelGGL(diag_setup_kernel, dim3(grid_for(c.nnodes)), dim3(kBlock), 0, c.stream,
                     (int)c.nnodes, c.node_dof.get(), c.node_fmask.get(), c.colptr.get(),
                     c.nzval.get(), c.diagpos.get(), c.diag.get(), c.fs.get());
  GH_CHECK_HIP(hipGetLastError());
  if (!c.fsai_ready) {
    DBuf<int> ovf;
    ovf.resize(1);
    GH_CHECK_HIP(hipMemsetAsync(ovf.get(), 0, sizeof(int), c.stream));
    hipLaunchKernelGGL(ell_index_kernel, dim3(grid_for(n)), dim3(kBlock), 0, c.stream, n,
                       c.colptr.get(), c.rowval.get(), c.diagpos.get(), c.gli.get(), c.gui.get(),
                       ovf.get());
    GH_CHECK_HIP(hipGetLastError());
    int h = 0;
    GH_CHECK_HIP(hipMemcpyAsync(&h, ovf.get(), sizeof(int), hipMemcpyDeviceToHost, c.stream));
    GH_CHECK_HIP(hipStreamSynchronize(c.stream));
    GH_REQUIRE(h == 0, GH_ERR_UNSUPPORTED, "FSAI rows longer than the 16-slot layout");
    c.fsai_ready = true;
  }
}

void mlp_sync_bf16(Ctx &c) {
  hipLaunchKernelGGL(to_bf16_kernel, dim3(grid_for(kMlpParams)), dim3(kBlock), 0, c.stream,
                     kMlpParams, c.params.get(), c.params_bf16.get());
  GH_CHECK_HIP(hipGetLastError());
}

void fsai_forward_build(Ctx &c, bool inference, bool solver) {
  GH_REQUIRE(c.have_mlp, GH_ERR_STATE, "no network weights: call gh_mlp_init or gh_mlp_set");
  fsai_prepare(c);
  const Lat3 L = lattice_of(c);
  const int C = (int)c.ncells;
  // K̂_aa of the box cell (every a), from the uploaded tabulation
  double kdiag = 0.0;
  {
    double det = c.sizes[0] * c.sizes[1] * c.sizes[2];
    for (int q = 0; q < c.nq; ++q) {
      double dot = 0.0;
      for (int d = 0; d < 3; ++d) {
        const double g = c.grad[(q * 8 + 0) * 3 + d] / c.sizes[d];
        dot += g * g;
      }
      kdiag += dot * std::fabs(det) * c.qw[q];
    }
  }
  const float logh = (float)(std::log(c.sizes[0] * c.sizes[1] * c.sizes[2]) / 3.0);
  hipStream_t s = c.stream;
  hipLaunchKernelGGL(features_kernel, dim3(grid_for(C)), dim3(kBlock), 0, s, L, (int64_t)C,
                     c.have_kappa ? c.kappa.get() : nullptr, c.node_dof.get(), c.diag.get(),
                     kdiag, logh, c.feat.get());
  if (inference) {
    const int ntiles = (C + 15) / 16;
    const unsigned grid =
        (unsigned)std::max(1, std::min((ntiles + kFwdWaves - 1) / kFwdWaves, 512));
    hipLaunchKernelGGL(mlp_fwd_mfma, dim3(grid), dim3(kFwdWaves * 64), 0, s, c.feat.get(),
                       c.params_bf16.get(), C, c.yo.get());
  } else {
    const unsigned grid = (unsigned)std::min((C + kTrainCells - 1) / kTrainCells, 2 * kTrainGrid);
    GH_CHECK_HIP(hipFuncSetAttribute((const void *)mlp_train_fwd,
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)sizeof(TrainLds)));  // past 64 KB
    hipLaunchKernelGGL(mlp_train_fwd, dim3(grid), dim3(256), sizeof(TrainLds), s, c.feat.get(),
                       c.params_bf16.get(), C, c.yo.get());
  }
  // box lattice: also the 14 lower-offset arrays of G for the stencil PCG kernels
  float *g14 = nullptr;
  if (c.box) {
    c.g14.resize((size_t)14 * std::max<int64_t>(c.nfree, 1));
    g14 = c.g14.get();
  }
  auto g_kern = inference ? g_assemble_kernel<false> : g_assemble_kernel<true>;
  hipLaunchKernelGGL(g_kern, dim3(grid_for(c.nnodes, 64)), dim3(64), 0, s, L, (int)c.nnodes,
                     c.node_dof.get(), c.node_fmask.get(), c.colptr.get(), c.yo.get(),
                     c.fs.get(), c.gl.get(), c.gu.get(), solver, c.gle.get(), c.gue.get(),
                     c.nfree, g14);
  GH_CHECK_HIP(hipGetLastError());
  c.fsai_built = solver;
}

namespace {

// One batch of NB probes from probe `first` on: loss partials and gĜ.
template <int NB>
void probe_batch(Ctx &c, uint64_t seed, int first, double coef) {
  hipStream_t s = c.stream;
  const int64_t n = c.nfree;
  const int32_t *cp = c.colptr.get(), *rv = c.rowval.get(), *dp = c.diagpos.get();
  const double *fs = c.fs.get();
  const uint8_t *sg = c.psign.get();
  const dim3 half(grid_for(n * kApplyLanes)), full(grid_for(n * kMultiLanes)), block(256);
  hipLaunchKernelGGL(rademacher_kernel, dim3(grid_for(n)), dim3(kBlock), 0, s, n, seed,
                     (uint64_t)first, NB, c.psign.get());
  // w = Gᵀ z, v = A w, r = z − G v, t = Gᵀ r, q = A t
  hipLaunchKernelGGL((apply_upper_kernel<NB, true>), half, block, 0, s, n, cp, rv, dp, c.gu.get(),
                     fs, sg, (const double *)nullptr, c.pw.get());
  hipLaunchKernelGGL(spmv_multi_kernel<NB>, full, block, 0, s, n, cp, rv, c.nzval.get(),
                     c.pw.get(), c.pv.get());
  hipLaunchKernelGGL(residual_kernel<NB>, dim3(kResidualBlocks), block, 0, s, n, cp, rv, dp,
                     c.gl.get(), fs, sg, c.pv.get(), c.pr.get(), c.lpart.get());
  hipLaunchKernelGGL((apply_upper_kernel<NB, false>), half, block, 0, s, n, cp, rv, dp,
                     c.gu.get(), fs, sg, c.pr.get(), c.pw.get());
  hipLaunchKernelGGL(spmv_multi_kernel<NB>, full, block, 0, s, n, cp, rv, c.nzval.get(),
                     c.pw.get(), c.pq.get());
  hipLaunchKernelGGL(pattern_grad_kernel<NB>, half, block, 0, s, n, cp, rv, dp, fs, c.pr.get(),
                     c.pv.get(), sg, c.pq.get(), coef, first > 0, c.gG.get());
  GH_CHECK_HIP(hipGetLastError());
}

__global__ void clear_kernel(int n, double *v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = 0.0;
}

}  // namespace

double fsai_train_step(Ctx &c, int nprobes, uint64_t seed, float lr) {
  GH_REQUIRE(nprobes >= 1 && nprobes <= 1024, GH_ERR_ARG, "nprobes must be in 1..1024");
  // a step that changes the weights leaves no factor for the solver: its copy is not written
  fsai_forward_build(c, false, !(lr > 0.0f));
  hipStream_t s = c.stream;
  const int64_t n = c.nfree;
  const int C = (int)c.ncells;
  const Lat3 L = lattice_of(c);
  // workspace of the training step, at its first one
  const size_t nv = (size_t)std::max<int64_t>(n, 1) * kProbeBatch;
  for (auto *b : {&c.pw, &c.pv, &c.pr, &c.pq}) b->resize(nv);
  c.psign.resize(std::max<int64_t>(n, 1));
  c.gG.resize(std::max<int64_t>(c.nnz, 1));
  c.lpart.resize(kResidualBlocks);
  c.dy.resize((size_t)C * kMlpOutPad);
  const int nb = std::min((C + kTrainCells - 1) / kTrainCells, kTrainGrid);
  c.wpart.resize((size_t)nb * kMlpParams);
  hipLaunchKernelGGL(clear_kernel, dim3(2), dim3(256), 0, s, kResidualBlocks, c.lpart.get());
  const double coef = -2.0 / ((double)nprobes * (double)std::max<int64_t>(n, 1));
  int k = 0;
  for (; k + 4 <= nprobes; k += 4) probe_batch<4>(c, seed, k, coef);
  if (k + 2 <= nprobes) {
    probe_batch<2>(c, seed, k, coef);
    k += 2;
  }
  if (k < nprobes) probe_batch<1>(c, seed, k, coef);
  hipLaunchKernelGGL(cell_grad_kernel, dim3(grid_for(C, 64)), dim3(64), 0, s, L, C,
                     c.node_dof.get(), c.node_fmask.get(), c.colptr.get(), c.gG.get(),
                     c.gl.get(), c.dy.get());
  GH_CHECK_HIP(hipGetLastError());
  // back-propagation (weights are the BF16 values the forward pass used), Adam
  const bool many = C > kTrainGrid * kRunTiles * kTrainCells;
  auto bwd = many ? mlp_train_bwd<true> : mlp_train_bwd<false>;
  const size_t bwd_lds = sizeof(TrainLds) + sizeof(TrainWeights) + (many ? 16 * 256 * 8 : 0);
  GH_CHECK_HIP(hipFuncSetAttribute((const void *)bwd, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)bwd_lds));
  hipLaunchKernelGGL(bwd, dim3(nb), dim3(256), bwd_lds, s, c.feat.get(), c.params_bf16.get(),
                     c.dy.get(), C, c.wpart.get());
  float b1t = 0.0f, b2t = 0.0f;
  if (lr > 0.0f) {
    ++c.adam_t;
    b1t = (float)std::pow(0.9, c.adam_t);
    b2t = (float)std::pow(0.999, c.adam_t);
  }
  hipLaunchKernelGGL(reduce_adam_kernel,
                     dim3(grid_for(kMlpParams, 256 / kReduceLanes)), dim3(256), 0, s,
                     c.wpart.get(), nb, c.grads.get(), lr, b1t, b2t, c.params.get(),
                     c.adam_m.get(), c.adam_v.get(), c.params_bf16.get());
  GH_CHECK_HIP(hipGetLastError());
  double lp[kResidualBlocks];
  HostCopy copy(c);
  copy.down(lp, c.lpart.get(), sizeof(lp));
  copy.finish();
  double loss = 0.0;
  for (int b = 0; b < kResidualBlocks; ++b) loss += lp[b];
  return loss / ((double)nprobes * (double)std::max<int64_t>(n, 1));
}

void grf_kappa(Ctx &c, int nmodes, const double *omega, const double *phase, double amp) {
  GH_REQUIRE(c.cartesian && c.dim == 3, GH_ERR_UNSUPPORTED,
             "the random-field coefficient is defined on a 3-D Cartesian mesh");
  GH_REQUIRE(nmodes >= 1 && nmodes <= 4096 && omega && phase, GH_ERR_ARG, "bad mode arrays");
  DBuf<double> dom, dph;
  dom.resize(3 * nmodes);
  dph.resize(nmodes);
  GH_CHECK_HIP(hipMemcpyAsync(dom.get(), omega, sizeof(double) * 3 * nmodes,
                              hipMemcpyHostToDevice, c.stream));
  GH_CHECK_HIP(hipMemcpyAsync(dph.get(), phase, sizeof(double) * nmodes, hipMemcpyHostToDevice,
                              c.stream));
  c.kappa.resize(c.ncells);
  const Lat3 L = lattice_of(c);
  hipLaunchKernelGGL(grf_kappa_kernel, dim3(grid_for(c.ncells)), dim3(kBlock), 0, c.stream, L,
                     c.ncells, c.origin[0], c.origin[1], c.origin[2], c.sizes[0], c.sizes[1],
                     c.sizes[2], nmodes, dom.get(), dph.get(), amp, c.kappa.get());
  GH_CHECK_HIP(hipGetLastError());
  GH_CHECK_HIP(hipStreamSynchronize(c.stream));
  c.have_kappa = true;
}

}  // namespace gh
